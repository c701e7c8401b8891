// Products of symmetric fp32 matrices that are kept as three bf16 planes each (hi = x rounded to the nearest bf16,
// mid = x - hi rounded, lo = x - hi - mid, which is exact: hi + mid + lo == x), for iterations whose every matrix is
// the result of such a product (the coupled Newton iteration of the inverse roots): the split is paid once per
// element in the epilogue of the product that makes it, not once per tile that reads it, and the k-loop is the
// direct-to-LDS loop of the rank-k kernels (syrk_dtl_tile.hpp) with nothing for the vector ALU to do.
//
//   C = A B  with A, B, C symmetric n x n:  C[i][j] = sum_k A[k][i] B[k][j],
// so both operand panels are [32 rows k][columns] blocks of a row-major matrix, exactly what that loop loads.  The
// six piece products that matter (see gemm_x3.hpp) are formed from the six plane panels of a k-tile, which are loaded
// once, smallest terms first; the accumulators of 8 k-tiles (256 k) are added to a running total and start again
// from zero, which keeps the rounding error of a long sum near that of one rounding.  Tiles on and above the diagonal are computed and mirrored, a diagonal tile from its upper
// triangle: the result is exactly symmetric, which the next product, reading it as its own transpose, relies on.  The epilogue splits the result into its planes and can, in the same pass, write the planes of
// c2_scale * C + c2_diag * I and fold max |C - I| into a device word (a NaN is kept, as torch.max keeps it).
//
// Storage of one matrix: three planes of n_pad x n_pad bf16, n_pad a multiple of the 192-wide tile, zero outside
// the n x n corner: products of padded matrices stay zero there, and no load or store needs a bounds test.  A plane
// is stored by blocks of 32 columns, [n_pad / 32][n_pad rows][32 columns] (plane_index): the 16 rows x 64 bytes that
// one wave-wide load brings into the LDS are then one contiguous kilobyte, eight whole cache lines, instead of
// sixteen half lines a row apart.
//
// Second form, two fp16 planes (NP = 2): hi = s x rounded to the nearest fp16, lo = s x - hi rounded, with a power
// of two s per matrix that the caller picks so that s |x| stays below the fp16 maximum.  hi + lo holds 22 bits of
// s x and everything down to 2^-25 absolutely (the matrix instruction takes fp16 denormals as they are): for a matrix
// whose entries are bounded, e.g. a polynomial of a normalised symmetric matrix, that is the accuracy of an fp32
// product, whose accumulation rounds at 2^-24 of the sum anyway, for three piece products (hi hi, hi lo, lo hi)
// instead of six and two thirds of the operand bytes.  The accumulators hold s_A s_B C; the epilogue multiplies by
// `in_unscale` = 1 / (s_A s_B) and writes the planes of c_scale C.
#pragma once
#include "gemm_f32.hpp"
#include "syrk_dtl_tile.hpp"

namespace ak {

constexpr int kPlaneTile = 192, kPlaneSmallTile = 64;
// Error words: a cache line each, kErrSlots per matrix.  All tiles of a matrix fold into theirs at once, and an atomic on a line
// that others are on takes 60 ns: with one word for the 91 tiles of 784 columns 5 us of the product.
constexpr int kErrStride = 16, kErrSlots = 16;
constexpr int kPlaneLdsBytes = 4 * 6 * 6 * 16 * 64;      // four stages of six plane panels of six [16 rows][64 bytes] blocks
constexpr int kPlaneMaxDim = 16128;      // 32-bit byte offsets inside a plane set, virtual k-tile numbers below 2^15
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// Number of a matrix buffer of an iteration: plain, or one of a pair (k, k + 1) of which an iteration reads one and writes the
// other; which one is decided on the device by the parity of the matrix's own step count.
struct PairedBuf {
  int16_t index, sel;       // sel 0: plain; 1: the one an iteration reads; 2: the one it writes; 3: 2 in a quartic step, else 1
};
// Kinds of a step (the caller's iteration; products that are the same in all of them name no kind).
enum StepKind { kStepPlain = 0, kStepLate = 1, kStepQuartic = 2 };
__device__ __forceinline__ int paired_buf(PairedBuf b, int parity, int kind = kStepPlain) {
  return b.index + (b.sel == 0 ? 0 : ((b.sel == 1 || (b.sel == 3 && kind != kStepQuartic)) ? parity : parity ^ 1));
}
// What the epilogue of a product makes of W = A B, element by element; U, P: elements of two further matrices.
//   kEpiPlain:   C = W, C2 = a I - b W (the next step's polynomial)
//   kEpiSquare:  C = 2 W - I, C2 = y_w W - y_w / 2 I + y_u U          (U = A = B)
//   kEpiQuartic: C = W + t_i I + t_u U + t_p P
//   kEpiShifted: C = W in plain steps, else W + t_i I + t_u U          (t_i, t_u of the call)
// Step table of a matrix, kCoefs floats a step: a, b, and of a quartic step y_u, y_w, t_i, t_u, t_p.
enum EpilogueKind { kEpiPlain = 0, kEpiSquare = 1, kEpiQuartic = 2, kEpiShifted = 3 };
constexpr int kEpiMatrices[4] = {0, 1, 2, 1};       // further matrices of an epilogue
constexpr int kCoefs = 8;
struct QuarticCoefs { float y_u, y_w, t_i, t_u, t_p; };
__device__ __forceinline__ QuarticCoefs quartic_coefs(const float* __restrict__ entry) {
  return QuarticCoefs{entry[2], entry[3], entry[4], entry[5], entry[6]};
}
// (every tile form rounds the same way: W enters last)
template <int EPI>
__device__ __forceinline__ float quartic_first(const QuarticCoefs& q, float w, float u, float pm, bool diagonal) {
  if constexpr (EPI == kEpiSquare) return __builtin_fmaf(2.f, w, diagonal ? -1.f : 0.f);
  const float shift = diagonal ? q.t_i : 0.f;
  return __builtin_fmaf(q.t_u, u, EPI == kEpiQuartic ? __builtin_fmaf(q.t_p, pm, shift) : shift) + w;
}
__device__ __forceinline__ float quartic_second(const QuarticCoefs& q, float w, float u, bool diagonal) {
  return __builtin_fmaf(q.y_w, w, __builtin_fmaf(q.y_u, u, diagonal ? -0.5f * q.y_w : 0.f));
}

struct PlaneGemm {
  __bf16* bufs;             // buffer i, plane set of batch entry z: bufs + i * buf_elems + z * set_elems (plane q: + q * plane_elems)
  int64_t buf_elems, set_elems;
  PairedBuf A, B, C, C2;    // C2.index < 0: no second result
  PairedBuf B_late;         // index >= 0: replaces B in steps other than plain ones
  PairedBuf U, P;           // of the epilogue, in the scale u_scale
  int epi;                  // EpilogueKind; kEpiSquare and kEpiQuartic run in quartic steps only
  float u_scale, shift_u, shift_i;
  const int* count;         // steps taken by each batch entry (the parity of its paired buffers)
  const int* accel;         // steps of each batch entry's table in front of the classical ones, where that decides the kind
  int early;                // of a step: plain before this one, quartic before accel, late behind it; 0: every step is plain
  const float* coef;        // entry's own table: C2 = a I - b C of step count + 1, the quartic's coefficients of step count
  int64_t coef_stride;
  int coef_last;            // steps beyond the table take its last entry
  float* errword;           // optional, kErrSlots words per batch entry, kErrStride apart
  const int* active;        // entry z runs only if active[z] != 0
  const float* settled;     // optional: entry z does not run where settled[z] > 0 (fp16 form)
  int* overflow;            // fp16 form: word z is set when a value of C or C2 does not fit the fp16 range
  int64_t plane_elems;      // n_pad * n_pad
  int n, n_pad, T;          // T = n_pad / tile
  // fp16 form only (powers of two): 1 / (scale of A's planes * scale of B's), scale of C's planes, scale of C2's
  float in_unscale, c_scale, c2_plane_scale;

  __device__ __forceinline__ int kind_of(int steps, int z) const {
    if (early == 0) return kStepPlain;
    const int quartic = accel[z];
    return quartic == 0 || steps < early ? kStepPlain : (steps < quartic ? kStepQuartic : kStepLate);
  }
};

// Element (i, j) of a plane stored by blocks of 32 columns.
__host__ __device__ __forceinline__ int64_t plane_index(int64_t i, int64_t j, int64_t n_pad) {
  return ((j >> 5) * n_pad + i) * 32 + (j & 31);
}

// The planes of x as 16-bit patterns.  NP = 3: bf16 hi, mid, lo (round to nearest each; the third remainder has at most
// 8 significant bits, so hi + mid + lo == x).  NP = 2: fp16 hi, lo of x, which the caller has scaled into range.
template <int NP>
__device__ __forceinline__ void plane_bits(float x, unsigned short (&o)[3]) {
  if constexpr (NP == 3) {
    const __bf16 hi = static_cast<__bf16>(x);
    const float r1 = x - static_cast<float>(hi);
    const __bf16 mid = static_cast<__bf16>(r1);
    const __bf16 lo = static_cast<__bf16>(r1 - static_cast<float>(mid));
    o[0] = __builtin_bit_cast(unsigned short, hi);
    o[1] = __builtin_bit_cast(unsigned short, mid);
    o[2] = __builtin_bit_cast(unsigned short, lo);
  } else {
    const _Float16 hi = static_cast<_Float16>(x);
    const _Float16 lo = static_cast<_Float16>(x - static_cast<float>(hi));
    o[0] = __builtin_bit_cast(unsigned short, hi);
    o[1] = __builtin_bit_cast(unsigned short, lo);
    o[2] = 0;
  }
}
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

// Wave (group q of GROUPS, block w of BLOCKS) holds chunk first + q of block w: every wave gets its 4 / GROUPS register quads
// of its block, the chunks first ... first + G - 1 (< chunks) added to `tot` in order.  part: 4 G BLOCKS KB of LDS that
// nothing else uses once all waves have arrived.
template <int BLOCKS, int GROUPS>
__device__ __forceinline__ void add_chunks(const floatx16& acc, floatx4 (&tot)[4 / GROUPS], int first, int chunks, int q, int w, int G,
                                           AK_LDS floatx4* part) {
  const int lane = threadIdx.x & 63;
  __syncthreads();
  if (q < G && first + q < chunks) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      part[((q * BLOCKS + w) * 4 + k) * 64 + lane] = floatx4{acc[4 * k], acc[4 * k + 1], acc[4 * k + 2], acc[4 * k + 3]};
  }
  __syncthreads();
  for (int c = 0; c < G && first + c < chunks; ++c) {
#pragma unroll
    for (int k = 0; k < 4 / GROUPS; ++k) {
      const floatx4 v = part[((c * BLOCKS + w) * 4 + q * (4 / GROUPS) + k) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) tot[k][e] += v[e];
    }
  }
}

// Two fp16 planes of four elements, times the inverse of their scale.
__device__ __forceinline__ floatx4 plane_values(u16x4 hi, u16x4 lo, float unscale) {
  floatx4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    v[e] = unscale * (static_cast<float>(__builtin_bit_cast(_Float16, static_cast<unsigned short>(hi[e]))) +
                      static_cast<float>(__builtin_bit_cast(_Float16, static_cast<unsigned short>(lo[e]))));
  return v;
}

// Epilogue of a quarter of a wave's 32 x 32 block of a 64 x 64 tile, rows 8 q + 4 g + e of it: planes of C (and of
// C2 = c2_scale C + c2_diag I), the mirror image of an off-diagonal tile, the lanes' largest |C - I| and whether all fits.
// EPI: see EpilogueKind; u, pm: the quarter's elements of the further matrices.
template <int NP, int EPI>
__device__ __forceinline__ void plane_epilogue(const PlaneGemm& p, int ti, int tj, int z, int wr, int wc, int q, floatx4 sum,
                                               int parity, int kind, float c2_diag, float c2_scale, const QuarticCoefs& qc,
                                               floatx4 u, floatx4 pm, float& vmax, bool& fits) {
  const int lane = threadIdx.x & 63, g = lane >> 5, l32 = lane & 31;
  const int i0 = ti * kPlaneSmallTile, j0 = tj * kPlaneSmallTile;
  unsigned short* __restrict__ sets = reinterpret_cast<unsigned short*>(p.bufs) + static_cast<int64_t>(z) * p.set_elems;
  unsigned short* __restrict__ C = sets + paired_buf(p.C, parity, kind) * p.buf_elems;
  unsigned short* __restrict__ C2 = p.C2.index >= 0 ? sets + paired_buf(p.C2, parity, kind) * p.buf_elems : nullptr;
  const bool off_diag = ti != tj;
  const float unscale = NP == 2 ? p.in_unscale : 1.f, cs = NP == 2 ? p.c_scale : 1.f, c2s = NP == 2 ? p.c2_plane_scale : 1.f;
  const int gj = j0 + 32 * wc + l32, gi = i0 + 32 * wr + 8 * q + 4 * g;      // rows gi .. gi + 3
  u16x4 m1[NP], m2[NP];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float w = sum[e] * unscale;
    const bool inside = gi + e < p.n && gj < p.n, diagonal = gi + e == gj;
    float v = w;
    if constexpr (EPI == kEpiPlain) {
      if (inside && (off_diag || gi + e <= gj)) vmax = gemm_fold_absmax(vmax, v, diagonal, 1);
    } else {
      v = quartic_first<EPI>(qc, w, u[e], pm[e], diagonal && inside);
    }
    unsigned short o[3];
    if constexpr (NP == 2) fits = fits && fabsf(v * cs) <= 65504.f;      // (false for a NaN too)
    plane_bits<NP>(v * cs, o);
    // a diagonal tile keeps its upper triangle and mirrors it element by element: the next product reads
    // this matrix as its own transpose, which it has to be exactly
    const bool keep = off_diag || gi + e <= gj;
    const int64_t at = plane_index(gi + e, gj, p.n_pad);
    const int64_t mirror = plane_index(gj, gi + e, p.n_pad);
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      if (keep) C[s * p.plane_elems + at] = o[s];
      if (!off_diag && gi + e < gj) C[s * p.plane_elems + mirror] = o[s];
      m1[s][e] = o[s];
    }
    if (C2 != nullptr) {
      float x;
      if constexpr (EPI == kEpiPlain) x = c2_scale * v + ((diagonal && inside) ? c2_diag : 0.f);
      else x = quartic_second(qc, w, u[e], diagonal && inside);
      if constexpr (NP == 2) fits = fits && fabsf(x * c2s) <= 65504.f;
      plane_bits<NP>(x * c2s, o);
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        if (keep) C2[s * p.plane_elems + at] = o[s];
        if (!off_diag && gi + e < gj) C2[s * p.plane_elems + mirror] = o[s];
        m2[s][e] = o[s];
      }
    }
  }
  if (off_diag) {        // C[gj][gi .. gi + 3]: four consecutive elements of a row (gi is a multiple of 4)
    const int64_t at = plane_index(gj, gi, p.n_pad);
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      *reinterpret_cast<u16x4*>(C + s * p.plane_elems + at) = m1[s];
      if (C2 != nullptr) *reinterpret_cast<u16x4*>(C2 + s * p.plane_elems + at) = m2[s];
    }
  }
}

// The same epilogue for the 192-wide tile, through the LDS, which the k-loop has left free: the tile is written there
// transposed, [row j][4 consecutive i] as the accumulators hold it, and goes out as whole lines, 1 KB of consecutive bytes
// per wave and store: the mirror image as it lies, the tile itself through transposing reads (ds_read_b64_tr_b16).
// What bounds it: the burst of stores of all work groups at once.  As two-byte stores from the accumulators it took 59 us
// of a work group's 188 at 3072 columns (two results), and a third of every product; in this form 21 us (the clock of the
// device, which the products keep at its power limit, gives part of that back: 24 x 3072 122 -> 116 ms, 61 x 768 12.4 -> 10.5).  LDS rows of 64 bytes; their 8-byte chunks are permuted by the row (xor with row / 4), so that the 32 rows
// a wave writes at once fall into different banks.
// EPI other than plain (two planes): what a block of 32 x 32 needs of the further matrices is requested while the block before it
// is formed, transposed as the accumulators are: four elements of a row (the matrices are symmetric).
template <int NP, int EPI, class Sum>
__device__ __forceinline__ void plane_epilogue_wide(const PlaneGemm& p, int ti, int tj, int z, AK_LDS unsigned char* lds,
                                                    Sum sum) {
  static_assert(EPI == kEpiPlain || NP == 2, "further matrices in two planes");
  constexpr int FR = 3, WC = 2, TILE = kPlaneTile, BLOCK = TILE * 64, SLOT = 6 * BLOCK;      // one plane of the tile
  static_assert(2 * SLOT <= kPlaneLdsBytes, "two planes at a time");
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));       // (keeps the address arithmetic below the k-loop of the caller)
  asm volatile("" : "+s"(z));
  const int lane = tid & 63, wave = tid >> 6;
  const int wr = wave / WC, wc = wave % WC, g = lane >> 5, l32 = lane & 31;
  const int i0 = ti * TILE, j0 = tj * TILE;
  const int steps = p.count[z], parity = steps & 1, kind = NP == 2 ? p.kind_of(steps, z) : static_cast<int>(kStepPlain);
  unsigned short* __restrict__ sets = reinterpret_cast<unsigned short*>(p.bufs) + static_cast<int64_t>(z) * p.set_elems;
  const float* __restrict__ table = p.coef + static_cast<int64_t>(z) * p.coef_stride;
  float c2_diag = 0.f, c2_scale = 0.f;
  QuarticCoefs qc = {};
  if constexpr (EPI != kEpiPlain) {
    if constexpr (EPI == kEpiShifted) {
      if (kind != kStepPlain) qc = QuarticCoefs{0.f, 0.f, p.shift_i, p.shift_u, 0.f};
    } else {
      qc = quartic_coefs(table + kCoefs * min(steps, p.coef_last));
    }
  } else if (p.C2.index >= 0) {
    const float* __restrict__ next = table + kCoefs * min(steps + 1, p.coef_last);
    c2_diag = next[0];
    c2_scale = -next[1];
  }
  // elements of the further matrices: [parity of the block][matrix][quarter][plane]
  constexpr int AUX = kEpiMatrices[EPI];
  u16x4 aux[2][AUX > 0 ? AUX : 1][4][2] = {};
  auto load_aux = [&](int number) {
    if constexpr (AUX > 0) {
      if (number >= 9 || (EPI == kEpiShifted && kind == kStepPlain)) return;
      const int a = number / 3, b = number % 3;
      // element (gj, gi): gi in block of columns (i0 + 96 wr) / 32 + a of 32, 4 g further
      const uint32_t lane_at = (static_cast<uint32_t>((i0 >> 5) + FR * wr + a) * static_cast<uint32_t>(p.n_pad) + static_cast<uint32_t>(j0 + 32 * FR * wc + 32 * b + l32)) * 32u + 4u * g;
#pragma unroll
      for (int x = 0; x < AUX; ++x) {
        // (a uniform base and a 32-bit offset of the lane, which both planes share)
        const unsigned short* __restrict__ from = sets + paired_buf(x == 0 ? p.U : p.P, parity, kind) * p.buf_elems;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          aux[number & 1][x][q][0] = *reinterpret_cast<const u16x4*>(from + 8 * q + lane_at);
          aux[number & 1][x][q][1] = *reinterpret_cast<const u16x4*>(from + p.plane_elems + 8 * q + lane_at);
        }
      }
    }
  };
  const float aux_unscale = 1.f / p.u_scale;
  const bool off_diag = ti != tj, plain = off_diag && j0 + TILE <= p.n;       // (ti < tj: then the rows are inside too)
  const float unscale = NP == 2 ? p.in_unscale : 1.f, cs = NP == 2 ? p.c_scale : 1.f, c2s = NP == 2 ? p.c2_plane_scale : 1.f;
  float vmax = 0.f;
  bool fits = true;
  uint32_t vmax_bits = 0;             // the largest |C| / scale seen by plain tiles, as bits (those of a NaN are the largest)
  u16x4 upper = {0, 0, 0, 0};         // the largest magnitudes of the upper fp16 planes
  // address of element (row, col) of a transposed tile
  auto at = [](int row, int col) { return (col >> 5) * BLOCK + row * 64 + ((((col >> 2) & 7) ^ ((row >> 2) & 7)) << 3) + (col & 3) * 2; };

  // planes s0, s0 + 1 of one result into the LDS and from there to memory
  auto pass = [&](auto second_tag, auto s0_tag) {
    constexpr bool SECOND = decltype(second_tag)::value;
    constexpr int s0 = decltype(s0_tag)::value, COUNT = NP - s0 < 2 ? NP - s0 : 2;
    constexpr bool NEEDS = EPI == kEpiQuartic || EPI == kEpiShifted || (EPI == kEpiSquare && SECOND);      // of the further matrices
    if constexpr (NEEDS) load_aux(0);
    __syncthreads();
    // a tile on the diagonal or at the border of the matrix
    auto edge_block = [&](auto a_tag, auto b_tag) {
      constexpr int a = decltype(a_tag)::value, b = decltype(b_tag)::value, number = 3 * a + b;
      const int lj = 32 * FR * wc + 32 * b + l32, gj = j0 + lj;
      if constexpr (NEEDS) load_aux(number + 1);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int li = 32 * FR * wr + 32 * a + 8 * q + 4 * g, gi = i0 + li;      // rows gi .. gi + 3
        u16x4 m[COUNT];
        floatx4 u = {}, pm = {};
        if constexpr (NEEDS) u = plane_values(aux[number & 1][0][q][0], aux[number & 1][0][q][1], aux_unscale);
        if constexpr (AUX > 1) pm = plane_values(aux[number & 1][AUX - 1][q][0], aux[number & 1][AUX - 1][q][1], aux_unscale);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = sum(a, b, 4 * q + e) * unscale;
          const bool inside = gi + e < p.n && gj < p.n, diagonal = gi + e == gj;
          float x = v * cs;
          if constexpr (EPI != kEpiPlain) x = SECOND ? quartic_second(qc, v, u[e], diagonal && inside) * c2s
                                                     : quartic_first<EPI>(qc, v, u[e], pm[e], diagonal && inside) * cs;
          else if constexpr (SECOND) x = (c2_scale * v + ((diagonal && inside) ? c2_diag : 0.f)) * c2s;
          else if constexpr (s0 == 0)
            if (inside && (off_diag || gi + e <= gj)) vmax = gemm_fold_absmax(vmax, v, diagonal, 1);
          if constexpr (NP == 2) fits = fits && fabsf(x) <= 65504.f;      // (false for a NaN too)
          unsigned short o[3];
          plane_bits<NP>(x, o);
#pragma unroll
          for (int s = 0; s < COUNT; ++s) m[s][e] = o[s0 + s];
        }
        if (off_diag) {
#pragma unroll
          for (int s = 0; s < COUNT; ++s) *reinterpret_cast<AK_LDS u16x4*>(lds + s * SLOT + at(lj, li)) = m[s];
        } else {
          // a diagonal tile keeps its upper triangle and mirrors it element by element: the next product reads this
          // matrix as its own transpose, which it has to be exactly
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (li + e > lj) continue;
#pragma unroll
            for (int s = 0; s < COUNT; ++s) {
              *reinterpret_cast<AK_LDS unsigned short*>(lds + s * SLOT + at(lj, li + e)) = m[s][e];
              *reinterpret_cast<AK_LDS unsigned short*>(lds + s * SLOT + at(li + e, lj)) = m[s][e];
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);         // (values of other blocks split ahead would not fit the registers)
      }
    };
    // Every other tile needs no test per element.  The scales are powers of two but for c2_scale, whose product with them
    // is exact: one rounding, as above.  Two fp16 planes overflow where the upper one is infinite or a NaN.
    const float scale = SECOND ? c2_scale * (unscale * c2s) : unscale * cs;
    auto block = [&](auto a_tag, auto b_tag) {
#pragma clang fp contract(off)             // (x rounds before its planes are taken, as in the other tiles: the same bits)
      constexpr int a = decltype(a_tag)::value, b = decltype(b_tag)::value, number = 3 * a + b;
      const int lj = 32 * FR * wc + 32 * b + l32;
      if constexpr (NEEDS) load_aux(number + 1);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int li = 32 * FR * wr + 32 * a + 8 * q + 4 * g;
        u16x4 m[COUNT];
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = sum(a, b, 4 * q + e) * scale;
        if constexpr (EPI != kEpiPlain) {
          floatx4 u = {}, pm = {};
          if constexpr (NEEDS) u = plane_values(aux[number & 1][0][q][0], aux[number & 1][0][q][1], aux_unscale);
          if constexpr (AUX > 1) pm = plane_values(aux[number & 1][AUX - 1][q][0], aux[number & 1][AUX - 1][q][1], aux_unscale);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = sum(a, b, 4 * q + e) * unscale;
            x[e] = SECOND ? quartic_second(qc, v, u[e], false) * c2s : quartic_first<EPI>(qc, v, u[e], pm[e], false) * cs;
          }
        }
        if constexpr (EPI == kEpiPlain && !SECOND && s0 == 0) {
          if (p.errword != nullptr) {
#pragma unroll
            for (int e = 0; e < 4; ++e) vmax_bits = max(vmax_bits, __builtin_bit_cast(uint32_t, x[e]) & 0x7fffffffu);
          }
        }
        if constexpr (NP == 2) {
          typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
          typedef float f32x4 __attribute__((ext_vector_type(4)));
          const f32x4 xv = {x[0], x[1], x[2], x[3]};
          const f16x4 hi = __builtin_convertvector(xv, f16x4);
          const f16x4 lo = __builtin_convertvector(xv - __builtin_convertvector(hi, f32x4), f16x4);
          m[0] = __builtin_bit_cast(u16x4, hi);
          m[1] = __builtin_bit_cast(u16x4, lo);
          upper = __builtin_elementwise_max(upper, m[0] & (unsigned short)0x7fff);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            unsigned short o[3];
            plane_bits<NP>(x[e], o);
#pragma unroll
            for (int s = 0; s < COUNT; ++s) m[s][e] = o[s0 + s];
          }
        }
#pragma unroll
        for (int s = 0; s < COUNT; ++s) *reinterpret_cast<AK_LDS u16x4*>(lds + s * SLOT + at(lj, li)) = m[s];
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto blocks = [](auto&& f) {
      using J0 = std::integral_constant<int, 0>;
      using J1 = std::integral_constant<int, 1>;
      using J2 = std::integral_constant<int, 2>;
      f(J0{}, J0{}); f(J0{}, J1{}); f(J0{}, J2{});
      f(J1{}, J0{}); f(J1{}, J1{}); f(J1{}, J2{});
      f(J2{}, J0{}); f(J2{}, J1{}); f(J2{}, J2{});
    };
    if (plain) blocks(block);
    else blocks(edge_block);
    __syncthreads();
    unsigned short* __restrict__ out = sets + paired_buf(SECOND ? p.C2 : p.C, parity, kind) * p.buf_elems + s0 * p.plane_elems;
    // A wave takes rows 16 (wave + 4 t), t < 3, of every block of 32 columns; all its LDS addresses and all its memory
    // addresses differ by constants of the wave.
    {   // rows gj, columns gi: lane = row l / 4 of 16, 16 bytes l % 4
      const int row = 16 * wave + (lane >> 2), col = 8 * (lane & 3);
      AK_LDS const unsigned char* lo = lds + at(row, col);
      AK_LDS const unsigned char* hi = lds + at(row, col + 4);
      const uint32_t lane_off = (lane >> 2) * 32 + col;
#pragma unroll
      for (int s = 0; s < COUNT; ++s)
#pragma unroll 2
        for (int blk = 0; blk < 6; ++blk) {
          unsigned short* dst = out + s * p.plane_elems + plane_index(j0 + 16 * wave, i0 + 32 * blk, p.n_pad);
#pragma unroll
          for (int t = 0; t < 3; ++t) {
            const u16x4 x = *reinterpret_cast<AK_LDS const u16x4*>(lo + s * SLOT + blk * BLOCK + t * 4096);
            const u16x4 y = *reinterpret_cast<AK_LDS const u16x4*>(hi + s * SLOT + blk * BLOCK + t * 4096);
            *reinterpret_cast<u16x8*>(dst + t * 2048 + lane_off) = u16x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
          }
        }
    }
    if (off_diag) {
      // rows gi, columns gj: lane (t4, j16) takes row j16 of 16 and columns 8 t4 .. 8 t4 + 7 of a block, two transposing reads
      const int t4 = lane >> 4, j16 = lane & 15, c = 16 * wave + 4 * (j16 & 3);
      AK_LDS const unsigned char* lo = lds + at(8 * t4 + (j16 >> 2), c);
      AK_LDS const unsigned char* hi = lds + at(8 * t4 + 4 + (j16 >> 2), c);
      const uint32_t lane_off = j16 * 32 + 8 * t4;
#pragma unroll
      for (int s = 0; s < COUNT; ++s)
#pragma unroll 2
        for (int blk = 0; blk < 6; ++blk) {
          unsigned short* dst = out + s * p.plane_elems + plane_index(i0 + 16 * wave, j0 + 32 * blk, p.n_pad);
#pragma unroll
          for (int t = 0; t < 3; ++t) {
            const int off = s * SLOT + blk * 2048 + t * 2 * BLOCK;
            const short4v x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((AK_LDS short4v*)(lo + off));
            const short4v y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((AK_LDS short4v*)(hi + off));
            *reinterpret_cast<short8v*>(dst + t * 2048 + lane_off) = short8v{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
          }
        }
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S2 = std::integral_constant<int, 2>;
  pass(std::false_type{}, S0{});
  if constexpr (NP == 3) pass(std::false_type{}, S2{});
  if ((EPI == kEpiPlain || EPI == kEpiSquare) && p.C2.index >= 0) {
    pass(std::true_type{}, S0{});
    if constexpr (NP == 3) pass(std::true_type{}, S2{});
  }
  if (plain) {
    vmax = __builtin_bit_cast(float, vmax_bits) * (1.f / cs);             // (a power of two)
    fits = NP != 2 || max(max(upper[0], upper[1]), max(upper[2], upper[3])) < 0x7c00;
  }
  if (p.errword != nullptr)
    gemm_store_absmax(p.errword + (static_cast<int64_t>(z) * kErrSlots + (ti + tj) % kErrSlots) * kErrStride, vmax, lane);
  if (NP == 2 && !fits) atomicOr(p.overflow + z, 1);
}

// One 192 x 192 tile (ti <= tj) of batch entry z.  4 waves (2 x 2), 3 x 3 blocks of 32 x 32 per wave.
// A k-tile is 16 rows of all six planes (three of A's column block ti, three of B's column block tj): 36 KB of LDS per
// stage, four stages.  Per k-tile and wave: 6 pairs of planes x 9 matrix instructions, 9 wave-wide 16-byte loads (a
// load fills the 16 rows x 64 bytes of one 32-column block), one barrier.  The loads run two and a half k-tiles ahead
// (what they miss in the L2 takes microseconds to arrive); the barrier sits in the middle of a k-tile, so that the
// second half can already read the first fragments of the next one.
__device__ __forceinline__ void plane_tile(const PlaneGemm& p, int ti, int tj, int z) {
  constexpr int WR = 2, WC = 2, FR = 3, FC = 3, NCB = 6, BK = 16, S = 4;
  constexpr int BT = 32 * FR * WR;
  constexpr int BLOCK = BK * 64;                   // one 32-column block of one plane: [16 rows][64 bytes]
  constexpr int PANEL = NCB * BLOCK;               // one plane of one operand's 192 columns
  constexpr int STAGE = 6 * PANEL;                 // planes 0..2 of A's panel, then planes 0..2 of B's
  constexpr int LOADS = 6 * NCB / (WR * WC);       // wave-wide loads per wave and k-tile
  constexpr int CHUNK = 16;                        // k-tiles per partial sum (256 k)
  static_assert(BT == kPlaneTile && S * STAGE == kPlaneLdsBytes, "tile geometry");
  extern __shared__ __attribute__((aligned(1024))) unsigned char dtl_smem[];
  AK_LDS unsigned char* lds = (AK_LDS unsigned char*)dtl_smem;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const int steps = p.count[z], parity = steps & 1;
  if (p.active[z] == 0 || (steps == 0 && p.C.index == 0)) return;      // (buffer 0 of the first step is given)

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave / WC, wc = wave % WC;
  const int nk = p.n_pad / BK;
  const uint32_t plane_bytes = static_cast<uint32_t>(p.plane_elems) * 2u;

  u32x4 rsrc[2];
#pragma unroll
  for (int P = 0; P < 2; ++P) {
    const uint64_t ba = reinterpret_cast<uint64_t>(p.bufs + paired_buf(P == 0 ? p.A : p.B, parity) * p.buf_elems +
                                                   static_cast<int64_t>(z) * p.set_elems);
    rsrc[P][0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(ba));
    rsrc[P][1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(ba >> 32) & 0xffffu);
    rsrc[P][2] = kDtlRange;
    rsrc[P][3] = 0x00020000u;
  }

  // The 36 blocks of a k-tile (operand P, plane q, column block cb) are dealt to the waves round-robin: wave w loads
  // blocks w, w + 4, ...; lane l brings row l / 4, 16-byte chunk l % 4 of the block's rows.
  // one block of one k-tile is 1 KB of consecutive bytes of the plane: block column (6 ti + cb), rows 16 kt ..
  const uint32_t lane_off = static_cast<uint32_t>(lane) * 16u;
  const uint32_t colblock_bytes = static_cast<uint32_t>(p.n_pad) * 64u;
  auto issue_load = [&](int kt, int stage, int l) {
    const uint32_t r = static_cast<uint32_t>(kt * BK) * 64u + lane_off;
    const int blk = wave + 4 * l;                  // 0 .. 35 = (P * 3 + q) * 6 + cb
    const int P = blk / 18, q = (blk / 6) % 3, cb = blk % 6;
    const uint32_t col = static_cast<uint32_t>((P == 0 ? ti : tj) * NCB + cb) * colblock_bytes;
    // (P differs between the waves of one instruction slot: both descriptors, one select)
    const u32x4 d = P == 0 ? rsrc[0] : rsrc[1];
    load_to_lds(d, lds0 + stage * STAGE + blk * BLOCK, kt < nk ? r + q * plane_bytes + col : 0u);
  };
  auto issue_loads = [&](int kt, int stage) {
#pragma unroll
    for (int l = 0; l < LOADS; ++l) issue_load(kt, stage, l);
  };

  floatx16 acc[FR][FC], tot[FR][FC];
#pragma unroll
  for (int a = 0; a < FR; ++a)
#pragma unroll
    for (int b = 0; b < FC; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) tot[a][b][r] = 0.f;

  const int g = lane >> 5, hl = (lane >> 4) & 1, j16 = lane & 15;
  const int frag_lane = (8 * g + (j16 >> 2)) * 64 + hl * 32 + (j16 & 3) * 8;
  AK_LDS const unsigned char* fragI = lds + frag_lane + wr * FR * BLOCK;
  AK_LDS const unsigned char* fragJ = lds + frag_lane + wc * FC * BLOCK + 3 * PANEL;

  auto tr = [](AK_LDS const unsigned char* q) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((AK_LDS short4v*)(q));
  };
  // A group = the FR (FC) fragments of one plane of A's (B's) panel for one k-tile.
  auto read_a = [&](bf16x8 (&f)[FR], int soff, int plane, int blk) {
    AK_LDS const unsigned char* q = fragI + soff + plane * PANEL + blk * BLOCK;
    f[blk] = pack_bf16x8(tr(q), tr(q + 256));
  };
  auto read_b = [&](bf16x8 (&f)[FC], int soff, int plane, int blk) {
    AK_LDS const unsigned char* q = fragJ + soff + plane * PANEL + blk * BLOCK;
    f[blk] = pack_bf16x8(tr(q), tr(q + 256));
  };
  bf16x8 fa[3][FR], fb[3][FC], fb0_next[FC];
  // The nine matrix instructions of one pair of planes, with the three fragment reads of a group that a later pair
  // needs spread between them (what: 0 none, 1 plane `plane` of A into fa[plane], 2 plane `plane` of B into fb[plane],
  // 3 plane 0 of B into fb0_next).
  // first_load >= 0: loads first_load .. first_load + 2 of k-tile load_kt go out one by one between the matrix
  // instructions (a wave alone on its SIMD cannot afford the issue time of nine in a row)
  auto pair_step = [&](const bf16x8 (&ca)[FR], const bf16x8 (&cb)[FC], auto what_tag, auto plane_tag, int soff,
                       int first_load = -1, int load_kt = 0) {
    constexpr int WHAT = decltype(what_tag)::value, PLANE = decltype(plane_tag)::value;
#pragma unroll
    for (int m = 0; m < FR * FC; ++m) {
      const int a = m / FC, b = m % FC;
      acc[a][b] = mfma_bf16(ca[a], cb[b], acc[a][b]);
      if (first_load >= 0 && m % 3 == 0) {
        __builtin_amdgcn_sched_barrier(0);
        issue_load(load_kt, load_kt & (S - 1), first_load + m / 3);
      }
      if (WHAT != 0 && m % 3 == 1) {
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (WHAT == 1) read_a(fa[PLANE], soff, PLANE, m / 3);
        if constexpr (WHAT == 2) read_b(fb[PLANE], soff, PLANE, m / 3);
        if constexpr (WHAT == 3) read_b(fb0_next, soff, 0, m / 3);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  // One k-tile: the six pairs in an order in which every step needs one new group only, smallest products first and
  // (hi, hi) last: (lo, hi), (mid, hi), (mid, mid), (hi, mid), (hi, lo), (hi, hi).  On entry fa[2] and b0 hold the
  // k-tile's first two groups; the last two steps fetch those of the next k-tile (plane 0 of B is in use until the
  // end, so it alternates between two register sets).
  auto ktile = [&](int kt, const bf16x8 (&b0)[FC], auto next_b0_tag) {
    constexpr int NEXT_B0 = decltype(next_b0_tag)::value;      // 2: into fb[0], 3: into fb0_next
    const int soff = (kt & (S - 1)) * STAGE, soff_next = ((kt + 1) & (S - 1)) * STAGE;
    pair_step(fa[2], b0, I1{}, I1{}, soff);
    pair_step(fa[1], b0, I2{}, I1{}, soff);
    pair_step(fa[1], fb[1], I1{}, I0{}, soff);
    // k-tile kt + 1 has landed for this wave (the loads of kt + 2 may still fly), then for all; and all waves are
    // done with k-tile kt - 1, whose stage the loads of k-tile kt + 3 fill
    wait_vmcnt<LOADS>();
    __syncthreads();
    pair_step(fa[0], fb[1], I2{}, I2{}, soff, 0, kt + 3);
    pair_step(fa[0], fb[2], I1{}, I2{}, soff_next, 3, kt + 3);
    if constexpr (NEXT_B0 == 3) pair_step(fa[0], b0, I3{}, I0{}, soff_next, 6, kt + 3);
    else pair_step(fa[0], b0, I2{}, I0{}, soff_next, 6, kt + 3);
  };

  issue_loads(0, 0);
  issue_loads(1, 1);
  issue_loads(2, 2);
  wait_vmcnt<2 * LOADS>();
  __syncthreads();
#pragma unroll
  for (int blk = 0; blk < 3; ++blk) { read_a(fa[2], 0, 2, blk); read_b(fb[0], 0, 0, blk); }
  // chunks of CHUNK k-tiles, each summed from zero and then added to the running total (two nested loops: with one
  // loop and a conditional reset the accumulators change register file at every k-tile)
  for (int kt0 = 0; kt0 < nk; kt0 += CHUNK) {
#pragma unroll
    for (int a = 0; a < FR; ++a)
#pragma unroll
      for (int b = 0; b < FC; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
    const int kt1 = kt0 + CHUNK < nk ? kt0 + CHUNK : nk;      // (n_pad is a multiple of 192: an even number of k-tiles)
    for (int kt = kt0; kt < kt1; kt += 2) {
      ktile(kt, fb[0], I3{});
      ktile(kt + 1, fb0_next, I2{});
    }
#pragma unroll
    for (int a = 0; a < FR; ++a)
#pragma unroll
      for (int b = 0; b < FC; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[a][b][r] += acc[a][b][r];
  }
  wait_vmcnt<0>();                                             // the loads past the last k-tile, before the LDS is released

  plane_epilogue_wide<3, kEpiPlain>(p, ti, tj, z, lds, [&](int a, int b, int r) { return tot[a][b][r]; });
}

// The same tile on two fp16 planes per operand.  A k-tile is 16 rows of four plane panels (24 KB per stage, six
// stages: the loads run four and a half k-tiles ahead), three pairs of planes x 9 matrix instructions per wave:
// (lo, hi), (hi, hi), (hi, lo).  On entry fa[1] and fb[0] hold the k-tile's first two groups; the first two steps read
// the other two, the last one the first two groups of the next k-tile.
template <int EPI>
__device__ __forceinline__ void plane_tile_h2(const PlaneGemm& p, int ti, int tj, int z) {
  constexpr int WR = 2, WC = 2, FR = 3, FC = 3, NCB = 6, BK = 16, S = 6;
  constexpr int BT = 32 * FR * WR;
  constexpr int BLOCK = BK * 64;
  constexpr int PANEL = NCB * BLOCK;
  constexpr int STAGE = 4 * PANEL;                 // planes 0..1 of A's panel, then planes 0..1 of B's
  constexpr int LOADS = 4 * NCB / (WR * WC);
  constexpr int CHUNK = 16;
  static_assert(BT == kPlaneTile && S * STAGE == kPlaneLdsBytes, "tile geometry");
  extern __shared__ __attribute__((aligned(1024))) unsigned char dtl_smem[];
  AK_LDS unsigned char* lds = (AK_LDS unsigned char*)dtl_smem;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const int steps = p.count[z], parity = steps & 1, kind = p.kind_of(steps, z);
  if (p.active[z] == 0 || (steps == 0 && p.C.index == 0)) return;      // (buffer 0 of the first step is given)
  if ((EPI == kEpiSquare || EPI == kEpiQuartic) && kind != kStepQuartic) return;
  if (p.settled != nullptr && p.settled[z] > 0.f) return;
  const PairedBuf B = p.B_late.index >= 0 && kind != kStepPlain ? p.B_late : p.B;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave / WC, wc = wave % WC;
  const int nk = p.n_pad / BK;
  const uint32_t plane_bytes = static_cast<uint32_t>(p.plane_elems) * 2u;

  u32x4 rsrc[2];
#pragma unroll
  for (int P = 0; P < 2; ++P) {
    const uint64_t ba = reinterpret_cast<uint64_t>(p.bufs + paired_buf(P == 0 ? p.A : B, parity, kind) * p.buf_elems +
                                                   static_cast<int64_t>(z) * p.set_elems);
    rsrc[P][0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(ba));
    rsrc[P][1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(ba >> 32) & 0xffffu);
    rsrc[P][2] = kDtlRange;
    rsrc[P][3] = 0x00020000u;
  }
  // The 24 blocks of a k-tile (operand P, plane q, column block cb) are dealt to the waves round-robin.
  const uint32_t lane_off = static_cast<uint32_t>(lane) * 16u;
  const uint32_t colblock_bytes = static_cast<uint32_t>(p.n_pad) * 64u;
  auto issue_load = [&](int kt, int stage, int l) {
    const uint32_t r = static_cast<uint32_t>(kt * BK) * 64u + lane_off;
    const int blk = wave + 4 * l;                  // 0 .. 23 = (P * 2 + q) * 6 + cb
    const int P = blk / 12, q = (blk / 6) % 2, cb = blk % 6;
    const uint32_t col = static_cast<uint32_t>((P == 0 ? ti : tj) * NCB + cb) * colblock_bytes;
    const u32x4 d = P == 0 ? rsrc[0] : rsrc[1];
    load_to_lds(d, lds0 + stage * STAGE + blk * BLOCK, kt < nk ? r + q * plane_bytes + col : 0u);
  };
  auto issue_loads = [&](int kt, int stage) {
#pragma unroll
    for (int l = 0; l < LOADS; ++l) issue_load(kt, stage, l);
  };

  floatx16 acc[FR][FC], tot[FR][FC];
#pragma unroll
  for (int a = 0; a < FR; ++a)
#pragma unroll
    for (int b = 0; b < FC; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) tot[a][b][r] = 0.f;

  const int g = lane >> 5, hl = (lane >> 4) & 1, j16 = lane & 15;
  const int frag_lane = (8 * g + (j16 >> 2)) * 64 + hl * 32 + (j16 & 3) * 8;
  AK_LDS const unsigned char* fragI = lds + frag_lane + wr * FR * BLOCK;
  AK_LDS const unsigned char* fragJ = lds + frag_lane + wc * FC * BLOCK + 2 * PANEL;
  auto tr = [](AK_LDS const unsigned char* q) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((AK_LDS short4v*)(q));
  };
  bf16x8 fa[2][FR], fb[2][FC];                     // (fp16 patterns in 16-byte fragments)
  auto read_a = [&](int soff, int plane, int blk) {
    AK_LDS const unsigned char* q = fragI + soff + plane * PANEL + blk * BLOCK;
    fa[plane][blk] = pack_bf16x8(tr(q), tr(q + 256));
  };
  auto read_b = [&](int soff, int plane, int blk) {
    AK_LDS const unsigned char* q = fragJ + soff + plane * PANEL + blk * BLOCK;
    fb[plane][blk] = pack_bf16x8(tr(q), tr(q + 256));
  };
  using f16x8 = _Float16 __attribute__((ext_vector_type(8)));
  // what: 1 plane 0 of A, 2 plane 1 of B (both of this k-tile), 3 plane 1 of A and plane 0 of B of the next k-tile
  // first_load >= 0: loads first_load .. first_load + 2 of k-tile load_kt go out one by one between the matrix
  // instructions (a wave alone on its SIMD cannot afford the issue time of six in a row)
  auto pair_step = [&](const bf16x8 (&ca)[FR], const bf16x8 (&cb)[FC], auto what_tag, int soff, int first_load, int load_kt,
                       int load_stage) {
    constexpr int WHAT = decltype(what_tag)::value;
#pragma unroll
    for (int m = 0; m < FR * FC; ++m) {
      const int a = m / FC, b = m % FC;
      acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, ca[a]), __builtin_bit_cast(f16x8, cb[b]),
                                                         acc[a][b], 0, 0, 0);
      if (first_load >= 0 && m % 3 == 0) {
        __builtin_amdgcn_sched_barrier(0);
        issue_load(load_kt, load_stage, first_load + m / 3);
      }
      if (m % 3 == 1) {
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (WHAT == 1) read_a(soff, 0, m / 3);
        if constexpr (WHAT == 2) read_b(soff, 1, m / 3);
        if constexpr (WHAT == 3) read_a(soff, 1, m / 3);
      }
      if (WHAT == 3 && m % 3 == 2) {
        __builtin_amdgcn_sched_barrier(0);
        read_b(soff, 0, m / 3);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

#pragma unroll
  for (int t = 0; t < S - 1; ++t) issue_loads(t, t);
  wait_vmcnt<(S - 2) * LOADS>();
  __syncthreads();
#pragma unroll
  for (int blk = 0; blk < 3; ++blk) { read_a(0, 1, blk); read_b(0, 0, blk); }
  int stage = 0;                                   // kt % S
  for (int kt0 = 0; kt0 < nk; kt0 += CHUNK) {
#pragma unroll
    for (int a = 0; a < FR; ++a)
#pragma unroll
      for (int b = 0; b < FC; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
    const int kt1 = kt0 + CHUNK < nk ? kt0 + CHUNK : nk;
    for (int kt = kt0; kt < kt1; ++kt) {
      const int next = stage + 1 == S ? 0 : stage + 1, fill = stage == 0 ? S - 1 : stage - 1;
      const int soff = stage * STAGE, soff_next = next * STAGE;
      pair_step(fa[1], fb[0], I1{}, soff, -1, 0, 0);
      // k-tile kt + 1 has landed for this wave, then for all; and all waves are done with k-tile kt - 1, whose stage
      // the loads of k-tile kt + S - 1 fill
      wait_vmcnt<(S - 3) * LOADS>();
      __syncthreads();
      pair_step(fa[0], fb[0], I2{}, soff, 0, kt + S - 1, fill);
      pair_step(fa[0], fb[1], I3{}, soff_next, 3, kt + S - 1, fill);
      stage = next;
    }
#pragma unroll
    for (int a = 0; a < FR; ++a)
#pragma unroll
      for (int b = 0; b < FC; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[a][b][r] += acc[a][b][r];
  }
  wait_vmcnt<0>();
  plane_epilogue_wide<2, EPI>(p, ti, tj, z, lds, [&](int a, int b, int r) { return tot[a][b][r]; });
}

// A 64 x 64 tile (ti <= tj) for groups with too few 192-wide tiles to fill the device: 16 waves, of which group q = wave / 4
// sums the chunk of 256 k number q of every G (G = 4, 2, 1: as many as the matrix has chunks), its four waves one 32 x 32
// block each.  Every element is summed in the order of the 192-wide tile (piece products of 16 k, chunks of 256 k, the chunks
// in order through the LDS): the same bits, whichever tile a group takes.
// Bound by latencies one after the other: the launch with the way to the matrix's step count 4 us, the first operands 1.5, the
// ring 4 (S stages of 16 k per group keep 100 KB requested on the CU; the matrix instructions hide behind it), the sums 0.5,
// the two-byte stores and their way out of the L2 3 per result.  One product at 784 columns and four at 512 in one launch, two of them
// in one launch, one with a second result: 17.2, 28.8, 24.0 us with four waves a tile for all chunks, 14.5, 22.9, 18.7 so.
// Launches with more tiles than CUs take half as many waves and LDS a tile, two tiles to a CU.
template <int NP, int GROUPS> constexpr int kSmallTileStages = (NP == 2 ? 4 : 3) * GROUPS;          // of all groups together
template <int NP, int GROUPS> constexpr int kSmallTileLds = kSmallTileStages<NP, GROUPS> * 4 * NP * 1024;

// Waits until at most `stages` stages of LOADS loads are in flight (a constant once the caller's loop is unrolled).
template <int LOADS>
__device__ __forceinline__ void wait_loads(std::integral_constant<int, LOADS>, int stages) {
#define AK_WAIT(n) case n: wait_vmcnt<(n) * LOADS>(); break;
  switch (stages) {
    AK_WAIT(0) AK_WAIT(1) AK_WAIT(2) AK_WAIT(3) AK_WAIT(4) AK_WAIT(5) AK_WAIT(6) AK_WAIT(7) AK_WAIT(8) AK_WAIT(9) AK_WAIT(10)
    AK_WAIT(11) AK_WAIT(12) AK_WAIT(13) AK_WAIT(14)
    default: wait_vmcnt<0>();
  }
#undef AK_WAIT
}

template <int NP, int GROUPS, int G>
__device__ __forceinline__ void plane_tile_chunks(const PlaneGemm& p, int ti, int tj, int z, int parity, int kind,
                                                  AK_LDS unsigned char* lds, floatx4 (&tot)[4 / GROUPS]) {
  constexpr int BK = 16, BLOCK = BK * 64, STAGE = 4 * NP * BLOCK, S = kSmallTileStages<NP, GROUPS> / G, LOADS = NP, CHUNK = 256 / BK;
  static_assert((S - 1) * LOADS < 64 && kSmallTileLds<NP, GROUPS> >= G * 16384, "loads in flight; the chunks' sums");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave >> 2, w = wave & 3, wr = w >> 1, wc = w & 1;
  const int nk = p.n_pad / BK, chunks = (nk + CHUNK - 1) / CHUNK;
  const uint32_t plane_bytes = static_cast<uint32_t>(p.plane_elems) * 2u, colblock_bytes = static_cast<uint32_t>(p.n_pad) * 64u;
  const PairedBuf B = p.B_late.index >= 0 && kind != kStepPlain ? p.B_late : p.B;
  u32x4 rsrc[2];
#pragma unroll
  for (int P = 0; P < 2; ++P) {
    const uint64_t ba = reinterpret_cast<uint64_t>(p.bufs + paired_buf(P == 0 ? p.A : B, parity, kind) * p.buf_elems +
                                                   static_cast<int64_t>(z) * p.set_elems);
    rsrc[P][0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(ba));
    rsrc[P][1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(ba >> 32) & 0xffffu);
    rsrc[P][2] = kDtlRange;
    rsrc[P][3] = 0x00020000u;
  }
  AK_LDS unsigned char* ring = lds + group * S * STAGE;
  const uint32_t ring0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(ring));
  // block (operand P, plane q, column block cb) of a stage: 16 rows x 64 bytes, 1 KB of consecutive bytes
  auto issue = [&](int kt, int stage) {
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
      const int blk = w * LOADS + l, P = blk / (2 * NP), q = (blk / 2) % NP, cb = blk & 1;
      const uint32_t col = static_cast<uint32_t>(2 * (P == 0 ? ti : tj) + cb) * colblock_bytes;
      const u32x4 d = P == 0 ? rsrc[0] : rsrc[1];
      load_to_lds(d, ring0 + stage * STAGE + blk * BLOCK,
                  (kt < nk ? static_cast<uint32_t>(kt * BK) * 64u + q * plane_bytes + col : 0u) + lane * 16u);
    }
  };
  const int g = lane >> 5, hl = (lane >> 4) & 1, j16 = lane & 15;
  const int frag_lane = (8 * g + (j16 >> 2)) * 64 + hl * 32 + (j16 & 3) * 8;
  AK_LDS const unsigned char* fragI = ring + frag_lane + wr * BLOCK;
  AK_LDS const unsigned char* fragJ = ring + frag_lane + (2 * NP + wc) * BLOCK;
  auto frag = [](AK_LDS const unsigned char* q) {
    return pack_bf16x8(__builtin_amdgcn_ds_read_tr16_b64_v4i16((AK_LDS short4v*)(q)),
                       __builtin_amdgcn_ds_read_tr16_b64_v4i16((AK_LDS short4v*)(q + 256)));
  };
#pragma unroll
  for (int k = 0; k < 4 / GROUPS; ++k) tot[k] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int first = 0; first < chunks; first += G) {
    const int kt0 = (first + group) * CHUNK;
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    if (group < G) {
#pragma unroll
      for (int t = 0; t < S - 1 && t < CHUNK; ++t) issue(kt0 + t, t);
    }
#pragma unroll
    for (int t = 0; t < CHUNK; ++t) {
      // this wave's part of k-tile t has landed, then everybody's; and all are done with k-tile t - 1, whose stage the
      // next loads fill
      wait_loads(std::integral_constant<int, LOADS>{}, t + S - 2 < CHUNK ? S - 2 : CHUNK - 1 - t);
      __syncthreads();
      if (group < G) {
        if (t + S - 1 < CHUNK) issue(kt0 + t + S - 1, (t + S - 1) % S);
        if (kt0 + t < nk) {
          const int soff = (t % S) * STAGE;
          bf16x8 fa[NP], fb[NP];
#pragma unroll
          for (int q = 0; q < NP; ++q) {
            fa[q] = frag(fragI + soff + 2 * q * BLOCK);
            fb[q] = frag(fragJ + soff + 2 * q * BLOCK);
          }
          if constexpr (NP == 2) {
            acc = x3_mfma<true>(fa[1], fb[0], acc);
            acc = x3_mfma<true>(fa[0], fb[0], acc);
            acc = x3_mfma<true>(fa[0], fb[1], acc);
          } else {
            acc = mfma_bf16(fa[2], fb[0], acc);
            acc = mfma_bf16(fa[1], fb[0], acc);
            acc = mfma_bf16(fa[1], fb[1], acc);
            acc = mfma_bf16(fa[0], fb[1], acc);
            acc = mfma_bf16(fa[0], fb[2], acc);
            acc = mfma_bf16(fa[0], fb[0], acc);
          }
        }
      }
    }
    add_chunks<4, GROUPS>(acc, tot, first, chunks, group, w, G, reinterpret_cast<AK_LDS floatx4*>(lds));
    if (first + G < chunks) __syncthreads();               // the next round's loads overwrite the sums
  }
}

template <int NP, int GROUPS, int EPI>
__device__ __forceinline__ void plane_tile_small_epi(const PlaneGemm& p, int ti, int tj, int z, int steps, int kind, AK_LDS unsigned char* lds,
                                                     float& vmax, bool& fits) {
  const int chunks = (p.n_pad + 255) / 256, parity = steps & 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const float* __restrict__ table = p.coef + static_cast<int64_t>(z) * p.coef_stride;
  float c2_diag = 0.f, c2_scale = 0.f;                 // (under way while the product is formed, like the further matrices' elements)
  QuarticCoefs qc = {};
  constexpr int AUX = kEpiMatrices[EPI], QUADS = 4 / GROUPS;
  u16x4 aux[AUX > 0 ? AUX : 1][QUADS][2];
  if constexpr (EPI != kEpiPlain) {
    if constexpr (EPI == kEpiShifted) qc = QuarticCoefs{0.f, 0.f, p.shift_i, p.shift_u, 0.f};
    else qc = quartic_coefs(table + kCoefs * min(steps, p.coef_last));
    const unsigned short* sets = reinterpret_cast<const unsigned short*>(p.bufs) + static_cast<int64_t>(z) * p.set_elems;
    const int gj = tj * kPlaneSmallTile + 32 * (wave & 1) + (lane & 31);
    const int gi = ti * kPlaneSmallTile + 32 * ((wave >> 1) & 1) + 8 * (wave >> 2) * QUADS + 4 * (lane >> 5);
#pragma unroll
    for (int x = 0; x < AUX; ++x) {
      const unsigned short* from = sets + paired_buf(x == 0 ? p.U : p.P, parity, kind) * p.buf_elems + plane_index(gj, gi, p.n_pad);
#pragma unroll
      for (int k = 0; k < QUADS; ++k) {
        aux[x][k][0] = *reinterpret_cast<const u16x4*>(from + 8 * k);
        aux[x][k][1] = *reinterpret_cast<const u16x4*>(from + 8 * k + p.plane_elems);
      }
    }
  } else if (p.C2.index >= 0) {
    const float* __restrict__ next = table + kCoefs * min(steps + 1, p.coef_last);
    c2_diag = next[0];
    c2_scale = -next[1];
  }
  floatx4 sum[QUADS];
  if (GROUPS == 4 && chunks >= 3) plane_tile_chunks<NP, GROUPS, GROUPS>(p, ti, tj, z, parity, kind, lds, sum);
  else if (chunks >= 2) plane_tile_chunks<NP, GROUPS, 2>(p, ti, tj, z, parity, kind, lds, sum);
  else plane_tile_chunks<NP, GROUPS, 1>(p, ti, tj, z, parity, kind, lds, sum);
  const float aux_unscale = 1.f / p.u_scale;
#pragma unroll
  for (int k = 0; k < QUADS; ++k) {
    floatx4 u = {}, pm = {};
    if constexpr (AUX > 0) u = plane_values(aux[0][k][0], aux[0][k][1], aux_unscale);
    if constexpr (AUX > 1) pm = plane_values(aux[AUX - 1][k][0], aux[AUX - 1][k][1], aux_unscale);
    plane_epilogue<NP, EPI>(p, ti, tj, z, (wave >> 1) & 1, wave & 1, (wave >> 2) * QUADS + k, sum[k], parity, kind, c2_diag, c2_scale,
                            qc, u, pm, vmax, fits);
  }
}

template <int NP, int GROUPS>
__device__ __forceinline__ void plane_tile_small(const PlaneGemm& p, int ti, int tj, int z, int steps, int kind, AK_LDS unsigned char* lds,
                                                 float& vmax, bool& fits) {
  if constexpr (NP == 2) {
    if (p.epi == kEpiSquare) return plane_tile_small_epi<NP, GROUPS, kEpiSquare>(p, ti, tj, z, steps, kind, lds, vmax, fits);
    if (p.epi == kEpiQuartic) return plane_tile_small_epi<NP, GROUPS, kEpiQuartic>(p, ti, tj, z, steps, kind, lds, vmax, fits);
    if (p.epi == kEpiShifted && kind != kStepPlain)
      return plane_tile_small_epi<NP, GROUPS, kEpiShifted>(p, ti, tj, z, steps, kind, lds, vmax, fits);
  }
  plane_tile_small_epi<NP, GROUPS, kEpiPlain>(p, ti, tj, z, steps, kind, lds, vmax, fits);
}

// Tile number -> (ti <= tj), in bands of 8 tile columns, row by row inside a band: the 32 work groups that share an
// L2 at any time then work on about 4 rows x 8 columns of tiles, i.e. read 4 + 8 column panels between them instead
// of the 2 + 16 of two rows of the triangle.  Band c (columns 8c .. 8c + w - 1, w = 8 but for the last) holds 8c rows of
// w tiles above its diagonal block and w, w - 1, .. 1 tiles in the block; bands before it hold 32 c^2 + 4 c tiles.
__device__ __forceinline__ void decode_banded_tile(int id, int T, int& ti, int& tj) {
  int c = static_cast<int>((__builtin_sqrtf(1.f + 32.f * static_cast<float>(id)) - 1.f) * (1.f / 16.f));
  while (32 * (c + 1) * (c + 1) + 4 * (c + 1) <= id) ++c;
  while (32 * c * c + 4 * c > id) --c;
  const int w = T - 8 * c < 8 ? T - 8 * c : 8;
  int local = id - (32 * c * c + 4 * c);
  if (local < 8 * c * w) {
    ti = local / w;
    tj = 8 * c + local - ti * w;
    return;
  }
  local -= 8 * c * w;
  int r = 0;
  while (local >= w - r) { local -= w - r; ++r; }
  ti = 8 * c + r;
  tj = ti + local;
}

// grid: tiles on and above the diagonal x batch, XCD-contiguous
template <int NP, int EPI>
static __global__ __launch_bounds__(256) void plane_gemm_kernel(PlaneGemm p, int ntiles) {
  const uint32_t id = xcd_contiguous_id(blockIdx.x, gridDim.x);
  const int z = static_cast<int>(id / static_cast<uint32_t>(ntiles));
  int ti, tj;
  decode_banded_tile(static_cast<int>(id - static_cast<uint32_t>(z) * ntiles), p.T, ti, tj);
  if constexpr (NP == 3) plane_tile(p, ti, tj, z);
  else plane_tile_h2<EPI>(p, ti, tj, z);
}

// planes: 3 (bf16) or 2 (fp16, with the scales of PlaneGemm)
inline int launch_plane_gemm(const PlaneGemm& p, int planes, int batch, hipStream_t stream) {
  constexpr int kLds = kPlaneLdsBytes;
  if (p.n_pad % kPlaneTile != 0 || p.n_pad > kPlaneMaxDim || p.T * kPlaneTile != p.n_pad || batch <= 0 ||
      (planes != 2 && planes != 3) || (planes == 3 && p.epi != kEpiPlain))
    return AK_ERR_ARG;
  void (*const kernels[5])(PlaneGemm, int) = {plane_gemm_kernel<2, kEpiPlain>, plane_gemm_kernel<2, kEpiSquare>, plane_gemm_kernel<2, kEpiQuartic>,
                                              plane_gemm_kernel<2, kEpiShifted>, plane_gemm_kernel<3, kEpiPlain>};
  static bool attr_set = false;     // idempotent; a race sets it twice at worst
  if (!attr_set) {
    for (auto* k : kernels)
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
        return AK_ERR_LAUNCH;
    attr_set = true;
  }
  const int ntiles = p.T * (p.T + 1) / 2;
  hipLaunchKernelGGL(kernels[planes == 3 ? 4 : p.epi], dim3(static_cast<unsigned>(ntiles) * batch), dim3(256), kLds, stream, p, ntiles);
  return check_launch();
}

}  // namespace ak
