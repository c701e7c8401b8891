// Input factor A = U^T U of a 3 x 3 convolution with stride 1 and padding 1 on a channels-last bf16 input, from
// shifted correlations of the input instead of the unfolded matrix U (asdl/operations/conv.py:80-88 forms
// U U^T of the unfolded input; the result here is that matrix, summed in a different order).
//
// Block (t, t') of A, t = (ky, kx), is  sum over output positions o of  x[o + t - 1]^T x[o + t' - 1]  (x zero outside
// the image).  With p = o + t - 1 and D = t' - t that is  sum_p x[p]^T x[p + D]  over the pixels p whose output
// position lies inside the image.  The sum over ALL pixels, R_D, depends on the shift D only: 25 shifts, of which 13
// are distinct up to transposition (R_-D = R_D^T), replace the 45 distinct blocks, and each R_D is a product of the
// [N H W, C] pixel matrix with a row-shifted view of itself.  What R_D counts too often are the pixels p whose
// output position o = p - t + 1 falls outside the image: image row H-1 for ky = 0, row 0 for ky = 2, and the same
// for columns.  A pixel of such a row has p + D inside the image only if D_y = 0, so the corrections are
//   D_y = 0, ky != 1:            - S_row[r(ky)][D_x]      sums over one image row,    [N W] pixels
//   D_x = 0, kx != 1:            - S_col[q(kx)][D_y]      sums over one image column, [N H] pixels
//   D = 0, ky != 1 and kx != 1:  + K[r][q]                the corner pixel counted twice, [N] pixels
// 16 small matrices in all (2 rows x 3 shifts, 2 columns x 3 shifts, 4 corners).
//
// All 13 + 6 + 6 + 4 products are tiles of Gram matrices of "virtual" convolutions (stride 1, no padding at the top)
// and run on the direct-to-LDS tile of syrk_dtl_tile.hpp in ONE launch:
//   main    3 x 5 taps (dy = 0..2, dx = -2..2), positions = all pixels: rows [2C, 3C) (tap D = 0) times columns
//           [2C, 15C) (the 13 shifts (0,0..2), (1,-2..2), (2,-2..2)) of that Gram matrix;
//   rows    1 x 3 taps on the pixels of image row r;  columns  3 x 1 taps on the pixels of image column q;
//   corners 1 x 1 on the corner pixels.
// Every work group writes its accumulators as a partial tile; a second launch sums the partial tiles of the row
// splits in a fixed order into row-major matrices, a third assembles the dense factor in the (c, ky, kx) order,
// applying alpha and beta, with whole-line stores.  Executed matrix work: 26 M C^2 FLOP against 81 M C^2 for the
// upper triangle of U^T U.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <initializer_list>
#include <mutex>
#include <unordered_map>
#include "syrk_dtl_tile.hpp"

namespace ak {

constexpr int kCorrProds = 9;          // main, 2 image rows, 2 image columns, 4 corners
constexpr int kCorrShifts = 13;
constexpr int kCorrPieces = 29;        // [C, C] pieces of the reduced matrix: 13 shifts, 2 x 3 rows, 2 x 3 columns, 4 corners
constexpr int kCorrPiecesT = 25;       // of which the first 25 are also read transposed (the corners are symmetric)

struct CorrProd {
  const void* X;                       // first pixel of the product's positions
  int32_t M;                           // positions
  int32_t Ho, Wo, kw, KK, pw;          // virtual convolution (stride 1, no padding above)
  uint32_t mWo, mHo, mKw, mBlk;
  // Tiles: the row tap's C columns from tile ti0 on, `ntaps` column taps of C columns each from tile tj0 on.
  int32_t ti0, tj0, ntaps, tpt;        // tpt: tiles per tap in either direction (C / BT)
  int32_t kt_split, nsplit;            // k-tiles per row split, splits
  int32_t first_item, first_tile;      // running counts over the products
  int64_t part_off;                    // float4 index of partial tile (split 0, tile 0)
  int64_t out_off;                     // first column of the product in the reduced matrix red[C][29 C]
};

struct CorrArgs {
  CorrProd prod[kCorrProds];
  int32_t Cin, H, W, nprod;
  uint32_t mG;
  floatx4* part;
  float* red;
};

__device__ __forceinline__ int corr_find(const CorrArgs& a, int w, bool by_tile) {
  int pi = 0;
#pragma unroll
  for (int i = 1; i < kCorrProds; ++i)
    if (i < a.nprod && w >= (by_tile ? a.prod[i].first_tile : a.prod[i].first_item)) pi = i;
  return pi;
}

// Tile t of a product: (ti, tj) in the virtual Gram matrix, and (row, col) = where the tile starts in the product's
// [C, ntaps C] block of the reduced matrix, in tiles.
__device__ __forceinline__ void corr_tile_of(const CorrProd& cp, int t, int& ti, int& tj, int& row, int& col) {
  const int tap = t / (cp.tpt * cp.tpt), rem = t - tap * cp.tpt * cp.tpt;
  row = rem / cp.tpt;
  col = tap * cp.tpt + rem - row * cp.tpt;
  ti = cp.ti0 + row;
  tj = cp.tj0 + col;
}

__device__ __forceinline__ int corr_ntiles(const CorrProd& cp) { return cp.ntaps * cp.tpt * cp.tpt; }

// One work group per (product, row split, tile).
template <int WR, int WC, int FR, int FC>
__device__ __forceinline__ void corr_products_tile(const CorrArgs& a, uint32_t wg, uint32_t nwg) {
  constexpr int BT = DtlCfg<WR, WC, FR, FC, true>::BT;
  const int w = static_cast<int>(xcd_contiguous_id(wg, nwg));
  const CorrProd& cp = a.prod[corr_find(a, w, false)];
  DtlParams p{};
  p.X = cp.X;
  p.M = cp.M;
  p.d = static_cast<int64_t>(cp.KK) * a.Cin;
  p.Cin = a.Cin; p.H = a.H; p.W = a.W;
  p.kw = cp.kw; p.KK = cp.KK;
  p.sh = p.sw = 1; p.ph = 0; p.pw = cp.pw;
  p.Ho = cp.Ho; p.Wo = cp.Wo;
  p.G = a.Cin;
  p.mWo = cp.mWo; p.mHo = cp.mHo; p.mKw = cp.mKw; p.mBlk = cp.mBlk; p.mG = a.mG; p.mKK = 0;
  const int local = w - cp.first_item, ntiles = corr_ntiles(cp);
  const int s = local / ntiles, t = local - s * ntiles;
  int ti, tj, row, col;
  corr_tile_of(cp, t, ti, tj, row, col);
  const int64_t k_begin = static_cast<int64_t>(s) * cp.kt_split * kDtlBK;
  int64_t k_end = k_begin + static_cast<int64_t>(cp.kt_split) * kDtlBK;
  if (k_end > cp.M) k_end = cp.M;
  const int rows = k_begin < k_end ? static_cast<int>(k_end - k_begin) : 0;
  if (cp.nsplit == 1) {
    // the only split: the tile goes straight into the reduced matrix
    const int64_t ld = static_cast<int64_t>(kCorrPieces) * a.Cin;
    dtl_tile<WR, WC, FR, FC, true>(p, ti, tj, k_begin, rows, nullptr,
                                   a.red + cp.out_off + static_cast<int64_t>(row) * BT * ld + static_cast<int64_t>(col) * BT, ld);
    return;
  }
  floatx4* partial = a.part + cp.part_off + static_cast<int64_t>(local) * (BT * BT / 4);
  dtl_tile<WR, WC, FR, FC, true>(p, ti, tj, k_begin, rows, partial);
}

// Sums the partial tiles of the row splits (fixed order) into the product's columns of ONE row-major matrix
// red[C][29 C]: 13 C columns of the main product, 3 C per image row and image column, C per corner.
// grid (tiles of all products, 4 * FR * FC): one work group per float4 slot of every thread's accumulators.
template <int WR, int WC, int FR, int FC>
__device__ __forceinline__ void corr_reduce_tile(const CorrArgs& a, int tile, int slot) {
  constexpr int NW = WR * WC, BT = 32 * FR * WR;
  constexpr int64_t tile_f4 = BT * BT / 4;
  const CorrProd& cp = a.prod[corr_find(a, tile, true)];
  if (cp.nsplit == 1) return;                          // written by the product itself
  const int t = tile - cp.first_tile, ntiles = corr_ntiles(cp);
  int ti, tj, trow, tcol;
  corr_tile_of(cp, t, ti, tj, trow, tcol);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave / WC, wc = wave % WC, g = lane >> 5, l32 = lane & 31;
  const int q = slot & 3, b = (slot >> 2) % FC, aa = (slot >> 2) / FC;
  const floatx4* src = a.part + cp.part_off + t * tile_f4 + slot * (NW * 64) + tid;
  const int64_t stride = ntiles * tile_f4;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  int s = 0;
  for (; s + 8 <= cp.nsplit; s += 8) {                 // eight loads in flight, summed in pairs: 39 roundings in a row show
    floatx4 w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = src[(s + k) * stride];
    acc += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
  }
  for (; s < cp.nsplit; ++s) acc += src[s * stride];
  const int ld = kCorrPieces * a.Cin;
  const int row = trow * BT + 32 * FR * wr + 32 * aa + 8 * q + 4 * g;
  const int col = tcol * BT + 32 * FC * wc + 32 * b + l32;
  float* dst = a.red + cp.out_off + static_cast<int64_t>(row) * ld + col;
#pragma unroll
  for (int e = 0; e < 4; ++e) dst[static_cast<int64_t>(e) * ld] = acc[e];
}

// All products of one layer in one launch: one work group per (product, row split, tile).
template <int WR, int WC, int FR, int FC>
__global__ __launch_bounds__(WR * WC * 64) void corr_products_kernel(CorrArgs a) {
  corr_products_tile<WR, WC, FR, FC>(a, blockIdx.x, gridDim.x);
}

// grid (tiles of all products, 4 * FR * FC): one work group per float4 slot of every thread's accumulators.
template <int WR, int WC, int FR, int FC>
__global__ __launch_bounds__(WR * WC * 64) void corr_reduce_kernel(CorrArgs a) {
  corr_reduce_tile<WR, WC, FR, FC>(a, blockIdx.x, blockIdx.y);
}

// The dense factor from the reduced matrix.  One work group per block of CR channels of rows and 64 channels of
// columns: 9 CR x 576 elements.  A thread owns ONE result column (channel c2, tap t2) and walks down the rows, so
// a wave stores 64 consecutive floats of a row and the work group 576.  The [CR, 64] block of each of the 29 pieces
// and the [64, CR] block that the transposed shifts read are staged in the LDS first, all loads of a thread in
// flight at once.  For a fixed row tap t1 (a compile-time value in the unrolled loop) everything but the channel pair
// is a per-thread constant: which piece the element comes from, read straight or transposed, and which corrections
// apply.  Piece numbers: shift s = 5 dy + dx: s; image row e (0: first, 1: last), shift dx: 13 + 3 e + dx; image
// column e, shift dy: 19 + 3 e + dy; corner (r, q): 25 + 2 r + q.
struct CorrAsm {
  const float* red;
  float* A;
  int64_t lda;
  int32_t C;
  float alpha, beta;
};

constexpr int kAsmCC = 64;                      // channels of columns per work group
constexpr int kAsmThreads = 9 * kAsmCC;         // one thread per result column

template <int CR>
__global__ __launch_bounds__(kAsmThreads) void corr_assemble_kernel(CorrAsm a) {
  constexpr int FW = kAsmCC + 1, TW = CR + 1;            // row lengths of a straight / a transposed block
  constexpr int F = CR * FW, T = kAsmCC * TW;            // floats per block
  constexpr int SF = 0, ST = kCorrPieces * F;
  __shared__ float lds[kCorrPieces * F + kCorrPiecesT * T];
  const int tid = threadIdx.x, C = a.C;
  const int64_t ld = static_cast<int64_t>(kCorrPieces) * C;
  const int ci0 = blockIdx.y * CR, cj0 = blockIdx.x * kAsmCC;
  {
    // straight blocks: element (c1, c2) of piece pc is red[ci0 + c1][pc C + cj0 + c2]; consecutive threads read
    // consecutive c2.  transposed sources: red[cj0 + c2][pc C + ci0 + c1], consecutive threads consecutive c1.
    constexpr int NF = kCorrPieces * CR * kAsmCC, NT = kCorrPiecesT * CR * kAsmCC;
    constexpr int IF = (NF + kAsmThreads - 1) / kAsmThreads, IT = (NT + kAsmThreads - 1) / kAsmThreads;
    float vf[IF], vt[IT];
#pragma unroll
    for (int i = 0; i < IF; ++i) {
      const int idx = tid + i * kAsmThreads;
      const int c2 = idx % kAsmCC, c1 = (idx / kAsmCC) % CR, pc = idx / (kAsmCC * CR);
      vf[i] = idx < NF ? a.red[static_cast<int64_t>(ci0 + c1) * ld + pc * C + cj0 + c2] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int idx = tid + i * kAsmThreads;
      const int c1 = idx % CR, c2 = (idx / CR) % kAsmCC, pc = idx / (kAsmCC * CR);
      vt[i] = idx < NT ? a.red[static_cast<int64_t>(cj0 + c2) * ld + pc * C + ci0 + c1] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < IF; ++i) {
      const int idx = tid + i * kAsmThreads;
      const int c2 = idx % kAsmCC, c1 = (idx / kAsmCC) % CR, pc = idx / (kAsmCC * CR);
      if (idx < NF) lds[SF + pc * F + c1 * FW + c2] = vf[i];
    }
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int idx = tid + i * kAsmThreads;
      const int c1 = idx % CR, c2 = (idx / CR) % kAsmCC, pc = idx / (kAsmCC * CR);
      if (idx < NT) lds[ST + pc * T + c2 * TW + c1] = vt[i];
    }
  }
  __syncthreads();
  const int c2 = tid / 9, t2 = tid - 9 * c2, ky2 = t2 / 3, kx2 = t2 - 3 * ky2;
  float* dst = a.A + static_cast<int64_t>(ci0) * 9 * a.lda + static_cast<int64_t>(cj0) * 9 + tid;
  // where element (c1, this thread's c2) of piece pc lies: straight, or in the transposed block
  auto at_of = [&](int pc, bool straight, int& stride) {
    stride = straight ? FW : 1;
    return straight ? SF + pc * F + c2 : ST + pc * T + c2 * TW;
  };
#pragma unroll
  for (int t1 = 0; t1 < 9; ++t1) {
    const int ky = t1 / 3, kx = t1 % 3;
    const int dy = ky2 - ky, dx = kx2 - kx, s = dy * 5 + dx;
    const int adx = dx >= 0 ? dx : -dx, ady = dy >= 0 ? dy : -dy;
    // main term: shift s >= 0 is stored, s < 0 is the transpose of shift -s
    int m_st, r_st = 0, c_st = 0;
    const int m_at = at_of(s >= 0 ? s : -s, s >= 0, m_st);
    // corrections: the pixels of one image row / column have no output position under this row tap
    const int r = ky == 0 ? 1 : 0, q = kx == 0 ? 1 : 0;
    const bool use_r = ky != 1 && dy == 0, use_c = kx != 1 && dx == 0, use_k = ky != 1 && kx != 1 && s == 0;
    const int r_at = use_r ? at_of(13 + 3 * r + adx, dx >= 0, r_st) : 0;     // unused: a dummy read of lds[0]
    const int c_at = use_c ? at_of(19 + 3 * q + ady, dy >= 0, c_st) : 0;
    const int k_at = SF + (25 + 2 * r + q) * F + c2;
#pragma unroll
    for (int c1 = 0; c1 < CR; ++c1) {
      float v = lds[m_at + c1 * m_st];
      if (ky != 1) { const float x = lds[r_at + c1 * r_st]; v -= use_r ? x : 0.f; }
      if (kx != 1) { const float x = lds[c_at + c1 * c_st]; v -= use_c ? x : 0.f; }
      if (ky != 1 && kx != 1) { const float x = lds[k_at + c1 * FW]; v += use_k ? x : 0.f; }
      float* o = dst + static_cast<int64_t>(c1 * 9 + t1) * a.lda;
      v *= a.alpha;
      if (a.beta != 0.f) v += a.beta * *o;
      *o = v;
    }
  }
}

// ---- host side ------------------------------------------------------------------------------------------------

struct CorrPlan {
  CorrArgs args;            // X pointers, part and red are filled in per call
  int bt, items, tiles;
  size_t part_f4, red_floats;
  int64_t x_off[kCorrProds];   // byte offset of each product's first pixel from the tensor
};

static int corr_tile_width(int64_t C) {
  if (C % 256 == 0 && C >= 512) return 256;
  if (C % 128 == 0) return 128;
  if (C % 192 == 0) return 192;
  if (C % 64 == 0) return 64;
  return 0;
}

// ASDL_AMD_CONV_CORR=0 in the environment keeps the unfolded form for every layer (read once).
static bool corr_enabled() {
  static const bool on = [] {
    const char* v = std::getenv("ASDL_AMD_CONV_CORR");
    return !(v != nullptr && v[0] == '0');
  }();
  return on;
}

static bool corr_eligible(int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int ph, int pw) {
  if (!corr_enabled()) return false;
  if (kh != 3 || kw != 3 || sh != 1 || sw != 1 || ph != 1 || pw != 1) return false;
  if (corr_tile_width(C) == 0 || N <= 0 || H <= 0 || W <= 0) return false;
  if (N * H * W * C * 2 > static_cast<int64_t>(kDtlRange)) return false;          // 32-bit byte offsets
  if (N * H * W * (W > H ? W : H) >= (1ll << 32)) return false;                   // exact magic divisions
  if (15 * C * (15 * C + 256) >= (1ll << 32)) return false;
  return true;
}

static CorrPlan corr_plan_build(int64_t N, int64_t C, int64_t H, int64_t W) {
  CorrPlan pl{};
  const int bt = corr_tile_width(C);
  pl.bt = bt;
  const int cb = static_cast<int>(C / bt);
  const int occ = bt == 64 ? 4 : (bt == 128 ? 2 : 1);      // work groups per CU
  const int64_t slots = 256 * occ;
  CorrArgs& a = pl.args;
  a.Cin = static_cast<int32_t>(C); a.H = static_cast<int32_t>(H); a.W = static_cast<int32_t>(W);
  a.nprod = kCorrProds;
  a.mG = make_magic(static_cast<uint32_t>(C));
  auto fill = [&](int i, int64_t x_off, int64_t M, int64_t Ho, int64_t Wo, int kh_v, int kw_v, int pw_v, int ti0,
                  int tj0, int ntaps) {
    CorrProd& p = a.prod[i];
    pl.x_off[i] = x_off;
    p.M = static_cast<int32_t>(M);
    p.Ho = static_cast<int32_t>(Ho); p.Wo = static_cast<int32_t>(Wo);
    p.kw = kw_v; p.KK = kh_v * kw_v; p.pw = pw_v;
    p.mWo = make_magic(p.Wo); p.mHo = make_magic(p.Ho); p.mKw = make_magic(kw_v);
    p.mBlk = make_magic(static_cast<uint32_t>(C) * p.KK);
    p.ti0 = ti0; p.tj0 = tj0; p.ntaps = ntaps;
    p.tpt = cb;
  };
  const int64_t px = C * 2;                      // bytes per pixel
  fill(0, 0, N * H * W, H, W, 3, 5, 2, 2 * cb, 2 * cb, kCorrShifts);
  fill(1, 0, N * W, 1, W, 1, 3, 0, 0, 0, 3);                         // image row 0
  fill(2, (H - 1) * W * px, N * W, 1, W, 1, 3, 0, 0, 0, 3);          // image row H - 1
  fill(3, 0, N * H, H, 1, 3, 1, 0, 0, 0, 3);                         // image column 0
  fill(4, (W - 1) * px, N * H, H, 1, 3, 1, 0, 0, 0, 3);              // image column W - 1
  for (int r = 0; r < 2; ++r)
    for (int q = 0; q < 2; ++q)
      fill(5 + 2 * r + q, ((r ? H - 1 : 0) * W + (q ? W - 1 : 0)) * px, N, 1, 1, 1, 1, 0, 0, 0, 1);
  int items = 0, tiles = 0;
  size_t part = 0;
  int64_t red_col = 0;
  const size_t tile_f4 = static_cast<size_t>(bt) * bt / 4;
  for (int i = 0; i < kCorrProds; ++i) {
    CorrProd& p = a.prod[i];
    const int64_t ktiles = (p.M + kDtlBK - 1) / kDtlBK,
                  ntiles = static_cast<int64_t>(p.ntaps) * p.tpt * p.tpt;
    int64_t ns = 1;
    if (i == 0 && ntiles > 0) {
      // the main product fills the device once (the corrections ride in its tail); at least 8 k-tiles per split
      ns = (slots + ntiles / 2) / ntiles;
      const int64_t cap = ktiles / 8 < 1 ? 1 : ktiles / 8;
      if (ns > cap) ns = cap;
      if (ns < 1) ns = 1;
    } else if (i > 0) {
      ns = (ktiles + 15) / 16;          // corrections: chains of at most 16 k-tiles
    }
    p.kt_split = static_cast<int32_t>((ktiles + ns - 1) / ns);
    p.nsplit = static_cast<int32_t>((ktiles + p.kt_split - 1) / p.kt_split);
    p.first_item = items;
    p.first_tile = tiles;
    p.part_off = static_cast<int64_t>(part);
    p.out_off = red_col;
    red_col += static_cast<int64_t>(p.ntaps) * C;      // C per piece: 13 C, 3 C or C
    items += p.nsplit * static_cast<int>(ntiles);
    tiles += static_cast<int>(ntiles);
    part += static_cast<size_t>(p.nsplit) * ntiles * tile_f4;
  }
  pl.items = items;
  pl.tiles = tiles;
  pl.part_f4 = part;
  pl.red_floats = static_cast<size_t>(C) * kCorrPieces * C;       // red_col == 29 C
  return pl;
}

// Plans by shape.
template <class Plan>
struct CorrPlanCache {
  struct Key {
    int64_t N, C, H, W;
    bool operator==(const Key& o) const { return N == o.N && C == o.C && H == o.H && W == o.W; }
  };
  struct Hash {
    size_t operator()(const Key& k) const {
      uint64_t h = 0x9e3779b97f4a7c15ull;
      for (uint64_t v : {static_cast<uint64_t>(k.N), static_cast<uint64_t>(k.C), static_cast<uint64_t>(k.H),
                         static_cast<uint64_t>(k.W)})
        h = (h ^ v) * 0xff51afd7ed558ccdull + (h >> 29);
      return static_cast<size_t>(h);
    }
  };
  std::unordered_map<Key, Plan, Hash> plans;
  std::mutex lock;
  template <class Build>
  Plan find(int64_t N, int64_t C, int64_t H, int64_t W, Build&& build) {
    const Key key{N, C, H, W};
    std::lock_guard<std::mutex> guard(lock);
    auto it = plans.find(key);
    if (it != plans.end()) return it->second;
    if (plans.size() > 1024) plans.clear();
    const Plan plan = build();
    plans.emplace(key, plan);
    return plan;
  }
};

static CorrPlan corr_plan(int64_t N, int64_t C, int64_t H, int64_t W) {
  static CorrPlanCache<CorrPlan> cache;
  return cache.find(N, C, H, W, [&] { return corr_plan_build(N, C, H, W); });
}

static size_t corr_ws_layout(const CorrPlan& pl, size_t& red_at) {
  const size_t part_bytes = pl.part_f4 * sizeof(floatx4);
  red_at = (part_bytes + 255) & ~static_cast<size_t>(255);
  return red_at + pl.red_floats * sizeof(float);
}

template <int WR, int WC, int FR, int FC>
static int corr_launch_cfg(const CorrPlan& pl, const CorrArgs& args, hipStream_t stream) {
  using Cfg = DtlCfg<WR, WC, FR, FC, true>;
  auto kern = corr_products_kernel<WR, WC, FR, FC>;
  if (Cfg::LDS_BYTES > 64 * 1024) {
    static bool attr_set = false;     // idempotent; a race sets it twice at worst
    if (!attr_set) {
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                              Cfg::LDS_BYTES) != hipSuccess)
        return AK_ERR_LAUNCH;
      attr_set = true;
    }
  }
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(pl.items)), dim3(Cfg::NW * 64), Cfg::LDS_BYTES, stream, args);
  hipLaunchKernelGGL((corr_reduce_kernel<WR, WC, FR, FC>), dim3(static_cast<unsigned>(pl.tiles), 4 * FR * FC),
                     dim3(Cfg::NW * 64), 0, stream, args);
  return AK_OK;
}

size_t conv_corr_ws_bytes(int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int ph, int pw) {
  if (!corr_eligible(N, C, H, W, kh, kw, sh, sw, ph, pw)) return 0;
  size_t red_at;
  return corr_ws_layout(corr_plan(N, C, H, W), red_at);
}

// All products of the layer on the channels-last bf16 tensor x (C channels), reduced into red [C][29 C].
static int corr_products(const CorrPlan& plan, const void* x, floatx4* part, float* red, hipStream_t stream) {
  CorrPlan pl = plan;
  CorrArgs& args = pl.args;
  for (int i = 0; i < kCorrProds; ++i) args.prod[i].X = static_cast<const unsigned char*>(x) + pl.x_off[i];
  args.part = part;
  args.red = red;
  if (pl.bt == 64) return corr_launch_cfg<2, 2, 1, 1>(pl, args, stream);
  if (pl.bt == 128) return corr_launch_cfg<2, 2, 2, 2>(pl, args, stream);
  if (pl.bt == 192) return corr_launch_cfg<2, 2, 3, 3>(pl, args, stream);
  return corr_launch_cfg<2, 4, 4, 2>(pl, args, stream);
}

static int corr_assemble(const float* red, int64_t C, float alpha, float beta, float* A, int64_t lda, hipStream_t stream) {
  CorrAsm s{};
  s.red = red;
  s.A = A; s.lda = lda;
  s.C = static_cast<int32_t>(C);
  s.alpha = alpha; s.beta = beta;
  // channels of rows per work group: 4 (60 KB of LDS) where that still gives a work group per CU
  const dim3 block(kAsmThreads);
  if (C >= 256)
    hipLaunchKernelGGL((corr_assemble_kernel<4>), dim3(static_cast<unsigned>(C / kAsmCC), static_cast<unsigned>(C / 4)),
                       block, 0, stream, s);
  else if (C >= 128)
    hipLaunchKernelGGL((corr_assemble_kernel<2>), dim3(static_cast<unsigned>(C / kAsmCC), static_cast<unsigned>(C / 2)),
                       block, 0, stream, s);
  else
    hipLaunchKernelGGL((corr_assemble_kernel<1>), dim3(static_cast<unsigned>(C / kAsmCC), static_cast<unsigned>(C)),
                       block, 0, stream, s);
  return check_launch();
}

int conv_corr_syrk(const void* x, int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int ph,
                   int pw, float alpha, float beta, float* A, int64_t lda, void* ws, size_t ws_bytes,
                   hipStream_t stream) {
  if (!corr_eligible(N, C, H, W, kh, kw, sh, sw, ph, pw) || (reinterpret_cast<uintptr_t>(x) & 15) != 0)
    return AK_ERR_UNSUPPORTED;
  const CorrPlan pl = corr_plan(N, C, H, W);
  size_t red_at;
  const size_t need = corr_ws_layout(pl, red_at);
  if (ws == nullptr || ws_bytes < need) return AK_ERR_WORKSPACE;
  float* red = reinterpret_cast<float*>(static_cast<unsigned char*>(ws) + red_at);
  const int rc = corr_products(pl, x, static_cast<floatx4*>(ws), red, stream);
  if (rc != AK_OK) return rc;
  return corr_assemble(red, C, alpha, beta, A, lda, stream);
}

// ---- fp32 inputs: three bf16 planes ------------------------------------------------------------------------------
// An fp32 NCHW input takes the same path on the bf16 matrix cores at the accuracy of fp32 products: every element
// is split exactly into three bf16 pieces, x = hi + mid + lo (each the remainder rounded to the nearest bf16; the
// third needs no rounding), written channels-last, [hi | mid | lo] per pixel.  Six of the nine piece products count (the others
// are below 2^-24 of the product) and all of them belong to one element of the result: a work group brings the three planes of
// both operands into the LDS and sums them there, hi hi' on one accumulator, the five small ones on another.
// The planes lie in a frame of zeros, two columns in front of every image row and two rows behind every image: p + D of any
// shift D is a pixel or a zero, so that a shift is a constant added to an address and no load tests a border.
// Bound by the matrix instructions (24 per 16 pixels and wave, alone on its SIMD, with the LDS reads and the loads of the
// stages ahead between them) and by the operands' way into the LDS.  With the planes as 3 C channels of the products above, each
// piece product a tile of its own (all nine with 64 channels) and folded afterwards, all kernels of a layer took (128 samples)
//   64 x 32 x 32  217 us, now 125;  128 x 16 x 16  157, now 102;  256 x 8 x 8  175, now 106;  512 x 4 x 4  267, now 148
// (products alone 90, 74, 76 and 106), and the factor was twice as far from the one in 64 bits (9e-8 of its norm, now 4e-8).
// Two fp16 planes of channels scaled by powers of two would need half the matrix work, but hold 22 of the 24 bits: single products
// are off by up to 3.6e-7 instead of 1.2e-7.

constexpr int kC3K = 16;               // pixels of a stage
constexpr int kC3Stages = 4;

struct Corr3Prod {
  uint32_t base, sn, sy, sx;           // bytes: the first position's place in the planes, between images, rows, pixels of the positions
  int32_t M, Ho, Wo;                   // positions
  uint32_t mWo, mHo;
  int32_t ntaps, tiles_n;              // column taps of C columns each; tiles of columns
  int32_t kw;                          // of a window, whose taps are `pitch` bytes a row apart
  uint32_t pitch;
  int32_t k_split, nsplit;             // stages per split of the positions, splits
  int32_t first_item, first_tile;      // running counts over the products
  int64_t part_off;                    // float4 index of partial tile (split 0, tile 0)
  int64_t out_off;                     // first column of the product in the reduced matrix red[C][29 C]
  uint32_t toff[kCorrShifts];          // bytes from a position to its partner under each tap
};

struct Corr3Args {
  Corr3Prod prod[kCorrProds];
  const void* planes;
  uint32_t bytes;                      // of the planes: what lies behind them reads as zero
  int32_t C, tiles_m;
  floatx4* part;
  float* red;
};

// x: [N, C, H, W] fp32 -> planes: [N, Hp, Wp, 3 Cp] bf16, the image from (top, left) on in a frame of zeros (an image that does not fit
// is cut off), channels padded with zeros to Cp, a multiple of 32.  One work group per (sample, 32 pixels of the frame, 32 channels):
// coalesced reads along the pixels, 64-byte runs of channels per pixel and plane on the way out.
__global__ __launch_bounds__(256) void corr3_split_kernel(const float* __restrict__ x, uint16_t* __restrict__ planes, int C, int Cp, int H, int W, int Hp, int Wp,
                                                          int top, int left) {
  __shared__ float tile[32][33];
  const int n = blockIdx.z, p0 = blockIdx.x * 32, c0 = blockIdx.y * 32, px_all = Hp * Wp;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;          // 32 x 8
  const int at = p0 + tx, fy = at / Wp, row = fy - top, col = at - fy * Wp - left;
  const bool inside = at < px_all && row >= 0 && row < H && col >= 0 && col < W;
  const float* src = x + (static_cast<int64_t>(n) * C + c0) * H * W + (inside ? row * W + col : 0);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int c = ty + 8 * r;
    tile[c][tx] = inside && c0 + c < C ? src[static_cast<int64_t>(c) * H * W] : 0.f;
  }
  __syncthreads();
  uint16_t* dst = planes + (static_cast<int64_t>(n) * px_all + p0) * (3 * Cp) + c0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int px = ty + 8 * r;
    if (p0 + px >= px_all) continue;
    const float v = tile[tx][px];
    const __bf16 hi = static_cast<__bf16>(v);
    const float r1 = v - static_cast<float>(hi);
    const __bf16 mid = static_cast<__bf16>(r1);
    const __bf16 lo = static_cast<__bf16>(r1 - static_cast<float>(mid));
    uint16_t* q = dst + static_cast<int64_t>(px) * (3 * Cp) + tx;
    q[0] = __builtin_bit_cast(uint16_t, hi);
    q[Cp] = __builtin_bit_cast(uint16_t, mid);
    q[2 * Cp] = __builtin_bit_cast(uint16_t, lo);
  }
}

// Element (row, col) of a product's block of the reduced matrix.  Its first tap is the pixel itself: that piece is symmetric, and
// is made so exactly by its upper triangle.
__device__ __forceinline__ void corr3_store(const Corr3Args& a, const Corr3Prod& cp, int row, int col, float v) {
  if (col >= cp.ntaps * a.C) return;
  const int64_t ld = static_cast<int64_t>(kCorrPieces) * a.C;
  float* red = a.red + cp.out_off;
  if (col >= a.C) {
    red[row * ld + col] = v;
  } else if (row <= col) {
    red[row * ld + col] = v;
    red[col * ld + row] = v;
  }
}

// A tile wholly below the first tap's diagonal: its transpose writes it.
__device__ __forceinline__ bool corr3_below(const Corr3Args& a, int row0, int col0, int cols) { return row0 >= col0 + cols && col0 + cols <= a.C; }

__device__ __forceinline__ int corr3_find(const Corr3Args& a, int w, bool by_tile) {
  int pi = 0;
#pragma unroll
  for (int i = 1; i < kCorrProds; ++i)
    if (w >= (by_tile ? a.prod[i].first_tile : a.prod[i].first_item)) pi = i;
  return pi;
}

// Tile t of an upper triangle, its columns' tiles one after the other: the column of tiles.
__device__ __forceinline__ int corr3_column(int t) {
  int n = static_cast<int>((sqrtf(8.f * static_cast<float>(t) + 1.f) - 1.f) * 0.5f);
  n += (n + 1) * (n + 2) / 2 <= t;
  n -= n * (n + 1) / 2 > t;
  return n;
}

// One work group per (product, split of the positions, tile of 64 WR channels x 64 WC columns), four waves of 64 x 64.
// WINDOW: one product, of all taps with all taps, by the tiles of its upper triangle.
template <int WR, int WC, bool WINDOW>
__global__ __launch_bounds__(256, 1) void corr3_products_kernel(Corr3Args a) {
  constexpr int BR = 64 * WR, BC = 64 * WC, CBR = BR / 32, CBC = BC / 32, BLOCKS = 3 * (CBR + CBC);
  constexpr int LOADS = (BLOCKS + 3) / 4, STAGE = 4 * LOADS * 1024, S = kC3Stages, CHUNK = WINDOW ? 16 : 32;      // stages whose sums join a total
  static_assert(WR * WC == 4 && (!WINDOW || WR == WC), "four waves; two stages at a time");
  extern __shared__ __attribute__((aligned(1024))) unsigned char dtl_smem[];
  AK_LDS unsigned char* lds = (AK_LDS unsigned char*)dtl_smem;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave / WC, wc = wave % WC;
  // the main product's items, an XCD's in a row, then the corrections' in the tail (in one row, the last XCDs had all of those)
  const int first = WINDOW ? static_cast<int>(gridDim.x) : a.prod[1].first_item, blk0 = static_cast<int>(blockIdx.x);
  const int w = blk0 < first ? static_cast<int>(xcd_contiguous_id(blk0, first)) : blk0;
  const Corr3Prod& cp = a.prod[WINDOW ? 0 : corr3_find(a, w, false)];
  const int local = w - cp.first_item, ntiles = WINDOW ? a.tiles_m * (a.tiles_m + 1) / 2 : a.tiles_m * cp.tiles_n;
  const int split = local / ntiles, t = local - split * ntiles;
  int tn = t / a.tiles_m, tm = t - tn * a.tiles_m;
  if constexpr (WINDOW) {
    tn = corr3_column(t);
    tm = t - tn * (tn + 1) / 2;
  }
  const int row0 = tm * BR, col0 = tn * BC;
  if (!WINDOW && corr3_below(a, row0, col0, BC)) return;
  const int k0 = split * cp.k_split, k1 = min(k0 + cp.k_split, (cp.M + kC3K - 1) / kC3K);

  u32x4 rsrc;
  const uint64_t ba = reinterpret_cast<uint64_t>(a.planes);
  rsrc[0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(ba));
  rsrc[1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(ba >> 32) & 0xffffu);
  rsrc[2] = a.bytes;
  rsrc[3] = 0x00020000u;
  // A stage: blocks of [16 pixels][32 channels] (1 KB), those of A by plane and 32 channels, then those of B; dealt to the waves round-robin.
  // What a block adds to the address of its pixel:
  uint32_t block_at[LOADS];
#pragma unroll
  for (int l = 0; l < LOADS; ++l) {
    const int blk = wave + 4 * l;
    uint32_t at = kDtlOob;
    const bool of_a = blk < 3 * CBR;
    const int b = of_a ? blk : blk - 3 * CBR, blocks = of_a ? CBR : CBC, plane = b / blocks;
    const int col = (of_a ? row0 : col0) + 32 * (b % blocks), tap = col / a.C;
    if (blk < BLOCKS && tap < cp.ntaps) {
      at = static_cast<uint32_t>(plane * a.C + col - tap * a.C) * 2u;
      if constexpr (WINDOW) at += static_cast<uint32_t>(tap / cp.kw) * cp.pitch + static_cast<uint32_t>(tap % cp.kw) * static_cast<uint32_t>(6 * a.C);
      else at += of_a ? 0u : cp.toff[tap];
    }
    block_at[l] = __builtin_amdgcn_readfirstlane(at);
  }
  const int prow = lane >> 2;
  // byte offset of the lane's 16 bytes of its pixel of stage kt (kDtlOob: none), in parts without a branch (what they need is
  // held in scalar registers: read from memory in the loop, its latency stood in every stage)
  const auto held = [](uint32_t v) { return __builtin_amdgcn_readfirstlane(v); };
  const uint32_t M = held(min(cp.M, k1 * kC3K)), Wo = held(cp.Wo), Ho = held(cp.Ho), mWo = held(Wo == 1 ? 0 : cp.mWo), mHo = held(Ho == 1 ? 0 : cp.mHo);
  const uint32_t all_Wo = held(Wo == 1 ? ~0u : 0u), all_Ho = held(Ho == 1 ? ~0u : 0u), sn = held(cp.sn), sy = held(cp.sy), sx = held(cp.sx);
  const uint32_t base_lane = cp.base + (lane & 3) * 16u;
  struct Place { uint32_t pos, q1, n, at; };
  constexpr int PARTS = 6;
  auto place_part = [&](Place& p, int kt, int part) {
    if (part == 0) p.pos = static_cast<uint32_t>(kt * kC3K + prow), p.q1 = __umulhi(p.pos, mWo) | (p.pos & all_Wo);
    if (part == 1) p.n = __umulhi(p.q1, mHo) | (p.q1 & all_Ho);
    if (part == 2) p.at = base_lane + (p.pos - p.q1 * Wo) * sx;
    if (part == 3) p.at += p.n * sn;
    if (part == 4) p.at += (p.q1 - p.n * Ho) * sy;
    if (part == 5) p.at = p.pos < M ? p.at : kDtlOob;
  };
  auto load_one = [&](uint32_t pixel, int stage, int l) {
    const uint32_t at = pixel == kDtlOob || block_at[l] == kDtlOob ? kDtlOob : pixel + block_at[l];
    load_to_lds(rsrc, lds0 + stage * STAGE + (wave + 4 * l) * 1024, at);
  };

  floatx16 tot[2][2], big[2][2], small[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) tot[x][y][r] = 0.f;

  const int g = lane >> 5, hl = (lane >> 4) & 1, j16 = lane & 15;
  const int frag_lane = (8 * g + (j16 >> 2)) * 64 + hl * 32 + (j16 & 3) * 8;
  AK_LDS const unsigned char* frag_a = lds + frag_lane + 2 * wr * 1024;
  AK_LDS const unsigned char* frag_b = lds + frag_lane + (3 * CBR + 2 * wc) * 1024;
  auto tr = [](AK_LDS const unsigned char* q) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((AK_LDS short4v*)(q)); };
  struct Fragments { bf16x8 a[3][2], b[3][2]; };       // [plane][32 channels]
  // fragment u of twelve, in the order the matrix instructions want them: (lo, hi), (mid, hi), (mid, mid), (hi, mid), (hi, lo), (hi, hi)
  auto read_one = [&](Fragments& f, int soff, int u) {
    constexpr int PLANE[6] = {2, 0, 1, 1, 0, 2};
    constexpr bool OF_A[6] = {true, false, true, false, true, false};
    const int plane = PLANE[u >> 1], i = u & 1;
    AK_LDS const unsigned char* q = (OF_A[u >> 1] ? frag_a + plane * CBR * 1024 : frag_b + plane * CBC * 1024) + soff + i * 1024;
    (OF_A[u >> 1] ? f.a : f.b)[plane][i] = pack_bf16x8(tr(q), tr(q + 256));
  };
  // One stage: 24 matrix instructions on `now`; between them the fragments of the next stage, then the loads of the one S - 1 ahead.
  auto step = [&](int kt, int soff_next, int fill, const Fragments& now, Fragments& next) {
    wait_vmcnt<(S - 3) * LOADS>();             // stage kt + 1 has landed for this wave,
    __syncthreads();                           // then for all; and all have read stage kt
    Place p;
    constexpr int PA[6] = {2, 1, 1, 0, 0, 0}, PB[6] = {0, 0, 1, 1, 2, 0};
#pragma unroll
    for (int m = 0; m < 24; ++m) {
      const int pr = m >> 2, x = (m >> 1) & 1, y = m & 1;
      if (pr == 5) big[x][y] = mfma_bf16(now.a[PA[pr]][x], now.b[PB[pr]][y], big[x][y]);
      else small[x][y] = mfma_bf16(now.a[PA[pr]][x], now.b[PB[pr]][y], small[x][y]);
      __builtin_amdgcn_sched_barrier(0);
      if (m < 12) {
        read_one(next, soff_next, m);
        if (m & 1) place_part(p, kt + S - 1, m >> 1);
      } else if (m - 12 < LOADS) {
        load_one(p.at, fill, m - 12);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int s = 0; s < S - 1; ++s) {
    Place p;
#pragma unroll
    for (int part = 0; part < PARTS; ++part) place_part(p, k0 + s, part);
#pragma unroll
    for (int l = 0; l < LOADS; ++l) load_one(p.at, s, l);
  }
  wait_vmcnt<(S - 2) * LOADS>();
  __syncthreads();
  Fragments even, odd;
#pragma unroll
  for (int u = 0; u < 12; ++u) read_one(even, 0, u);
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) small[x][y][r] = 0.f;
  int stage = 0;                               // of k-tile kt; (the stages behind the last one hold zeros)
  for (int c = k0; c < k1; c += CHUNK) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int r = 0; r < 16; ++r) big[x][y][r] = 0.f;
    const int end = min(c + CHUNK, k1);
    for (int kt = c; kt < end; kt += 2) {
      step(kt, ((stage + 1) & (S - 1)) * STAGE, (stage + S - 1) & (S - 1), even, odd);
      step(kt + 1, ((stage + 2) & (S - 1)) * STAGE, (stage + S) & (S - 1), odd, even);
      stage = (stage + 2) & (S - 1);
    }
    // what a total rounds away goes to the small products' accumulator, which holds 2^-8 of the others and runs on to the end
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float t = tot[x][y][r], v = big[x][y][r], sum = t + v, more = sum - t;
          small[x][y][r] += (t - (sum - more)) + (v - more);
          tot[x][y][r] = sum;
        }
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (!__builtin_isinf(tot[x][y][r])) tot[x][y][r] += small[x][y][r];
  wait_vmcnt<0>();                             // the loads behind the last stage, before the LDS is released
  if (!WINDOW && cp.nsplit == 1) {
    const int l32 = lane & 31;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          corr3_store(a, cp, row0 + 64 * wr + 32 * x + 8 * (r >> 2) + 4 * g + (r & 3), col0 + 64 * wc + 32 * y + l32, tot[x][y][r]);
    return;
  }
  floatx4* part = a.part + cp.part_off + static_cast<int64_t>(local) * (BR * BC / 4) + tid;
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        part[((x * 2 + y) * 4 + q) * 256] = floatx4{tot[x][y][4 * q], tot[x][y][4 * q + 1], tot[x][y][4 * q + 2], tot[x][y][4 * q + 3]};
}

// Sums the partial tiles of the splits in a fixed order.  grid (tiles of all products, 16): one work group per float4 slot of every
// thread's accumulators.
template <int WR, int WC>
__global__ __launch_bounds__(256) void corr3_reduce_kernel(Corr3Args a) {
  constexpr int BR = 64 * WR, BC = 64 * WC;
  constexpr int64_t tile_f4 = BR * BC / 4;
  const Corr3Prod& cp = a.prod[corr3_find(a, blockIdx.x, true)];
  if (cp.nsplit == 1) return;                          // written by the product itself
  const int ntiles = a.tiles_m * cp.tiles_n, t = blockIdx.x - cp.first_tile, tn = t / a.tiles_m, tm = t - tn * a.tiles_m;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, slot = blockIdx.y;
  const int wr = wave / WC, wc = wave % WC, q = slot & 3, y = (slot >> 2) & 1, x = slot >> 3;
  if (corr3_below(a, tm * BR, tn * BC, BC)) return;
  const floatx4* src = a.part + cp.part_off + t * tile_f4 + slot * 256 + tid;
  const int64_t stride = ntiles * tile_f4;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};                // (in floats, these sums were the larger part of the result's error)
  int s = 0;
  for (; s + 8 <= cp.nsplit; s += 8) {                 // eight loads in flight
    floatx4 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = src[(s + k) * stride];
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += static_cast<double>(v[k][e]);
  }
  for (; s < cp.nsplit; ++s) {
    const floatx4 v = src[s * stride];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += static_cast<double>(v[e]);
  }
  const int row = tm * BR + 64 * wr + 32 * x + 8 * q + 4 * (lane >> 5), col = tn * BC + 64 * wc + 32 * y + (lane & 31);
#pragma unroll
  for (int e = 0; e < 4; ++e) corr3_store(a, cp, row + e, col, static_cast<float>(acc[e]));
}

struct Corr3Plan {
  Corr3Args args;                      // planes, part and red are filled in per call
  int items, tiles;
  bool wide;                           // 128 x 128 tiles, else 64 x 256
  size_t part_f4;
};

static int64_t corr3_pixel_bytes(int64_t C) { return 6 * C; }
static int64_t corr3_plane_bytes(int64_t N, int64_t C, int64_t H, int64_t W) { return N * (H + 2) * (W + 2) * corr3_pixel_bytes(C); }

// (the margin: what a shift of the last position adds)
static bool corr3_eligible(int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int ph, int pw) {
  return C % 64 == 0 && N <= 65535 && corr_eligible(N, 3 * C, H, W, kh, kw, sh, sw, ph, pw) &&
         corr3_plane_bytes(N, C, H, W) + 3 * (W + 2) * corr3_pixel_bytes(C) <= static_cast<int64_t>(kDtlRange);
}

static Corr3Plan corr3_plan_build(int64_t N, int64_t C, int64_t H, int64_t W) {
  Corr3Plan pl{};
  pl.wide = C % 128 == 0;
  const int64_t br = pl.wide ? 128 : 64, bc = pl.wide ? 128 : 256, px = corr3_pixel_bytes(C), Wp = W + 2, img = (H + 2) * Wp * px;
  Corr3Args& a = pl.args;
  a.bytes = static_cast<uint32_t>(corr3_plane_bytes(N, C, H, W));
  a.C = static_cast<int32_t>(C);
  a.tiles_m = static_cast<int32_t>(C / br);
  // kind of the taps: 0 the 13 shifts, 1 along the row, 2 along the column, 3 the pixel alone
  auto fill = [&](int i, int64_t first_px, int64_t M, int64_t Ho, int64_t Wo, int kind) {
    Corr3Prod& p = a.prod[i];
    p.base = static_cast<uint32_t>((first_px + 2) * px);
    p.sn = static_cast<uint32_t>(img); p.sy = static_cast<uint32_t>(Wp * px); p.sx = static_cast<uint32_t>(px);
    p.M = static_cast<int32_t>(M); p.Ho = static_cast<int32_t>(Ho); p.Wo = static_cast<int32_t>(Wo);
    p.mWo = make_magic(p.Wo); p.mHo = make_magic(p.Ho);
    p.ntaps = kind == 0 ? kCorrShifts : kind == 3 ? 1 : 3;
    p.tiles_n = static_cast<int32_t>((p.ntaps * C + bc - 1) / bc);
    for (int t = 0; t < p.ntaps; ++t) {
      const int dy = kind == 0 ? (t + 2) / 5 : kind == 2 ? t : 0, dx = kind == 0 ? t - 5 * dy : kind == 1 ? t : 0;
      p.toff[t] = static_cast<uint32_t>((dy * Wp + dx) * px);
    }
  };
  fill(0, 0, N * H * W, H, W, 0);
  for (int e = 0; e < 2; ++e) {
    fill(1 + e, e * (H - 1) * Wp, N * W, 1, W, 1);
    fill(3 + e, e * (W - 1), N * H, H, 1, 2);
    for (int q = 0; q < 2; ++q) fill(5 + 2 * e + q, e * (H - 1) * Wp + q * (W - 1), N, 1, 1, 3);
  }
  auto stages = [&](const Corr3Prod& p) { return static_cast<int64_t>(p.M + kC3K - 1) / kC3K; };
  // The main product in the number of splits (of at least 4 stages) and the corrections in chains of 32, 16 or 8 stages whose items end
  // first on the shader engine (8 CUs) that has most of both.  Items are dealt to the 32 engines in turn, and one whose engine is full holds up those
  // behind it: a 57th split of 128 x 64 x 32 x 32 leaves some engines no CU for their corrections.  In stages of the main product
  // (0.45 us): an item has 13 besides its own, a correction's stage (pixels an image or a row apart) is 1.25, the reduction of partial
  // tiles 10 and one per 20 tiles.  Splits and us, all kernels: 128 x 64 x 32 x 32: 48 124, 56 118, 57 130, 64 125;
  // 128 x 128 x 16 x 16: 10 123, 16 97, 18 106, 20 130; 128 x 256 x 8 x 8: 3 115, 4 100, 5 131, 8 106; 128 x 512 x 4 x 4: 1 139, 3 152.
  constexpr int64_t kEngines = 32, kCus = 8, kItem = 13;
  const int64_t main_tiles = static_cast<int64_t>(a.tiles_m) * a.prod[0].tiles_n, all = stages(a.prod[0]);
  auto chains = [&](const Corr3Prod& p, int64_t len) { return (stages(p) + len - 1) / len; };
  int64_t best = 1, best_chain = 32;
  double best_time = 0;
  for (int64_t chain : {32, 16, 8})
    for (int64_t ns = 1; ns <= std::max<int64_t>(1, std::min<int64_t>(all / 4, 2 * kEngines * kCus / main_tiles + 1)); ++ns) {
      const int64_t len = (all + ns - 1) / ns + kItem, n = main_tiles * ns, here = (n + kEngines - 1) / kEngines;
      int64_t busy[kCus], before = 0;    // (a heap of the times at which the CUs are free)
      for (int64_t c = 0; c < kCus; ++c) busy[c] = (here / kCus + (c < here % kCus)) * len;
      std::make_heap(busy, busy + kCus, std::greater<>());
      bool partial = ns > 1;
      for (int i = 1; i < kCorrProds; ++i) {
        const Corr3Prod& p = a.prod[i];
        const int64_t cs = chains(p, chain), after = before + a.tiles_m * p.tiles_n * cs, each = (stages(p) + cs - 1) / cs * 5 / 4 + kItem;
        int64_t count = (after + kEngines - 1) / kEngines - (before + kEngines - 1) / kEngines;
        for (int64_t& t : busy) t += count / kCus * each;
        for (count %= kCus; count > 0; --count) {
          std::pop_heap(busy, busy + kCus, std::greater<>());
          busy[kCus - 1] += each;
          std::push_heap(busy, busy + kCus, std::greater<>());
        }
        before = after;
        partial |= cs > 1;
      }
      const double time = static_cast<double>(*std::max_element(busy, busy + kCus)) + (partial ? 10.0 + 0.05 * static_cast<double>(n + before) : 0.0);
      if ((ns == 1 && chain == 32) || time < best_time) {
        best = ns;
        best_chain = chain;
        best_time = time;
      }
    }
  int items = 0, tiles = 0;
  size_t part = 0;
  int64_t red_col = 0;
  for (int i = 0; i < kCorrProds; ++i) {
    Corr3Prod& p = a.prod[i];
    const int64_t n = static_cast<int64_t>(a.tiles_m) * p.tiles_n, ns = i == 0 ? best : chains(p, best_chain);
    p.k_split = static_cast<int32_t>(((stages(p) + ns - 1) / ns + 1) / 2 * 2);        // (an even number of stages)
    p.nsplit = static_cast<int32_t>((stages(p) + p.k_split - 1) / p.k_split);
    p.first_item = items;
    p.first_tile = tiles;
    p.part_off = static_cast<int64_t>(part);
    p.out_off = red_col;
    red_col += p.ntaps * C;            // C per piece: 13 C, 3 C or C
    items += p.nsplit * static_cast<int>(n);
    tiles += static_cast<int>(n);
    if (p.nsplit > 1) part += static_cast<size_t>(p.nsplit * n * br * bc / 4);
  }
  pl.items = items;
  pl.tiles = tiles;
  pl.part_f4 = part;
  return pl;
}

static Corr3Plan corr3_plan(int64_t N, int64_t C, int64_t H, int64_t W) {
  static CorrPlanCache<Corr3Plan> cache;
  return cache.find(N, C, H, W, [&] { return corr3_plan_build(N, C, H, W); });
}

// [planes][partial tiles][red: C x 29 C]
static size_t corr3_layout(int64_t N, int64_t C, int64_t H, int64_t W, const Corr3Plan& pl, size_t& part_at, size_t& red_at) {
  auto aligned = [](size_t b) { return (b + 255) & ~static_cast<size_t>(255); };
  part_at = aligned(static_cast<size_t>(corr3_plane_bytes(N, C, H, W)));
  red_at = aligned(part_at + pl.part_f4 * sizeof(floatx4));
  return red_at + static_cast<size_t>(C) * kCorrPieces * C * sizeof(float);
}

size_t conv_corr_f32_ws_bytes(int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int ph, int pw) {
  if (!corr3_eligible(N, C, H, W, kh, kw, sh, sw, ph, pw)) return 0;
  size_t a, b;
  return corr3_layout(N, C, H, W, corr3_plan(N, C, H, W), a, b);
}

template <int WR, int WC>
static int corr3_launch(const Corr3Plan& pl, const Corr3Args& args, hipStream_t stream) {
  constexpr int kLds = kC3Stages * 4 * ((6 * (WR + WC) + 3) / 4) * 1024;
  static bool attr_set = false;     // idempotent; a race sets it twice at worst
  if (!attr_set) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(corr3_products_kernel<WR, WC, false>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
      return AK_ERR_LAUNCH;
    attr_set = true;
  }
  hipLaunchKernelGGL((corr3_products_kernel<WR, WC, false>), dim3(static_cast<unsigned>(pl.items)), dim3(256), kLds, stream, args);
  if (pl.part_f4 > 0)
    hipLaunchKernelGGL((corr3_reduce_kernel<WR, WC>), dim3(static_cast<unsigned>(pl.tiles), 16), dim3(256), 0, stream, args);
  return AK_OK;
}

int conv_corr_syrk_f32(const float* x, int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int ph,
                       int pw, float alpha, float beta, float* A, int64_t lda, void* ws, size_t ws_bytes,
                       hipStream_t stream) {
  if (!corr3_eligible(N, C, H, W, kh, kw, sh, sw, ph, pw)) return AK_ERR_UNSUPPORTED;
  const Corr3Plan pl = corr3_plan(N, C, H, W);
  size_t part_at, red_at;
  const size_t need = corr3_layout(N, C, H, W, pl, part_at, red_at);
  if (ws == nullptr || ws_bytes < need || (reinterpret_cast<uintptr_t>(ws) & 255) != 0) return AK_ERR_WORKSPACE;
  unsigned char* base = static_cast<unsigned char*>(ws);
  Corr3Args args = pl.args;
  args.planes = base;
  args.part = reinterpret_cast<floatx4*>(base + part_at);
  args.red = reinterpret_cast<float*>(base + red_at);
  hipLaunchKernelGGL(corr3_split_kernel, dim3(static_cast<unsigned>(((H + 2) * (W + 2) + 31) / 32), static_cast<unsigned>(C / 32), static_cast<unsigned>(N)),
                     dim3(256), 0, stream, x, reinterpret_cast<uint16_t*>(base), static_cast<int>(C), static_cast<int>(C), static_cast<int>(H), static_cast<int>(W),
                     static_cast<int>(H + 2), static_cast<int>(W + 2), 0, 2);
  const int rc = pl.wide ? corr3_launch<2, 2>(pl, args, stream) : corr3_launch<1, 4>(pl, args, stream);
  if (rc != AK_OK) return rc;
  return corr_assemble(args.red, C, alpha, beta, A, lda, stream);
}

// ---- other windows of fp32 inputs --------------------------------------------------------------------------------
// A strided window has no shifts to share: its factor is the product of all taps with all taps over the output positions, on the same
// planes and products, a tap another constant in the address of either operand.  The partial tiles lie in the order (tap, channel) of
// the columns; their sum, in double, is put into the factor's order (channel, tap) by the last kernel, which reads them once.  Totals are
// joined every 256 pixels, with what they round away: 3.0 to 4.9e-8 of the factor's norm from the one in 64 bits, the fp32 kernel's is
// 4.1 to 6.7e-8 over the same 26 windows.

// One work group per (32 channels of columns, 8 channels of rows, a tap of rows): 8 rows of 32 KK entries.  An entry is stored once, its
// row before its column; the other way round it is read transposed.
// (Many splits are few channels, and few work groups: a wave per tap of columns.)
__global__ __launch_bounds__(1024) void corr3_window_kernel(Corr3Args a, int KK, int C, float alpha, float beta, float* __restrict__ A, int64_t lda) {
  extern __shared__ float rows[];                      // [8][32 KK + 1]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, threads = blockDim.x, t = blockIdx.z;
  const int c0 = 8 * blockIdx.y, j0 = 32 * blockIdx.x, pitch = 32 * KK + 1, ntiles = a.tiles_m * (a.tiles_m + 1) / 2;
  const int nsplit = a.prod[0].nsplit;
  const int64_t stride = static_cast<int64_t>(ntiles) * 4096;
  // float4 of rows 4 (r / 4) ... + 3 of column c, of a tile on or above the diagonal
  auto place = [&](int r, int c) {
    const int tm = r >> 7, tn = c >> 7, x = (r >> 5) & 1, q = (r >> 3) & 3, g = (r >> 2) & 1, y = (c >> 5) & 1;
    return a.part + static_cast<int64_t>(tn * (tn + 1) / 2 + tm) * 4096 + ((x * 2 + y) * 4 + q) * 256 + (((r >> 6) & 1) * 2 + ((c >> 6) & 1)) * 64 + g * 32 + (c & 31);
  };
  for (int u = wave; u < KK; u += threads / 64) {
    const int p0 = t * a.C + c0, q0 = u * a.C + j0;    // first row, first column
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
    auto add = [&](const floatx4* src) {
      int s = 0;
      for (; s + 8 <= nsplit; s += 8) {                // eight loads in flight
        floatx4 v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = src[(s + k) * stride];
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[e] += static_cast<double>(v[k][e]);
      }
      for (; s < nsplit; ++s) {
        const floatx4 v = src[s * stride];
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] += static_cast<double>(v[e]);
      }
    };
    if ((p0 >> 5) < (q0 >> 5)) {
      const int g = lane >> 5, l32 = lane & 31;
      add(place(p0 + 4 * g, q0 + l32));
#pragma unroll
      for (int e = 0; e < 4; ++e) rows[(4 * g + e) * pitch + l32 * KK + u] = static_cast<float>(sum[e]);
    } else if ((p0 >> 5) > (q0 >> 5)) {
      const int r = 4 * (lane >> 3), c = lane & 7;
      add(place(q0 + r, p0 + c));
#pragma unroll
      for (int e = 0; e < 4; ++e) rows[c * pitch + (r + e) * KK + u] = static_cast<float>(sum[e]);
    } else {
      const int g = lane >> 5, l32 = lane & 31;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = p0 + 4 * g + e, j = q0 + l32, r = min(i, j);
        const float* src = reinterpret_cast<const float*>(place(r, max(i, j))) + (r & 3);
        double one = 0.0;
        for (int s = 0; s < nsplit; ++s) one += static_cast<double>(src[4 * s * stride]);
        rows[(4 * g + e) * pitch + l32 * KK + u] = static_cast<float>(one);
      }
    }
  }
  __syncthreads();
  const int width = min(32, C - j0) * KK;
  for (int r = 0; r < 8; ++r) {
    if (c0 + r >= C) return;
    float* __restrict__ dst = A + (static_cast<int64_t>(c0 + r) * KK + t) * lda + static_cast<int64_t>(j0) * KK;
    for (int j = tid; j < width; j += threads) {
      const float v = alpha * rows[r * pitch + j];
      dst[j] = beta != 0.f ? beta * dst[j] + v : v;
    }
  }
}

struct Corr3Window {
  int64_t Cp, Hp, Wp, Ho, Wo, plane_bytes;
  Corr3Args args;
  int items;
  size_t part_at, ws_bytes;
};

static bool corr3_window_plan(Corr3Window& v, int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int ph, int pw) {
  v = Corr3Window{};
  v.Ho = (H + 2 * ph - kh) / sh + 1;
  v.Wo = (W + 2 * pw - kw) / sw + 1;
  v.Cp = (C + 31) / 32 * 32;
  v.Hp = (v.Ho - 1) * sh + kh;
  v.Wp = (v.Wo - 1) * sw + kw;
  const int64_t px = 6 * v.Cp, KK = static_cast<int64_t>(kh) * kw, d = KK * v.Cp, M = N * v.Ho * v.Wo;
  if (!corr_enabled() || H + 2 * ph < kh || W + 2 * pw < kw || KK == 1 || KK > 32 || N > 65535 || v.Hp * v.Wp > (1 << 30) || d > 32768) return false;
  v.plane_bytes = N * v.Hp * v.Wp * px;
  if (v.plane_bytes + 64 * px > static_cast<int64_t>(kDtlRange) || (M + 1024) * std::max(v.Ho, v.Wo) >= (1ll << 32)) return false;
  Corr3Args& a = v.args;
  Corr3Prod& p = a.prod[0];
  a.bytes = static_cast<uint32_t>(v.plane_bytes);
  a.C = static_cast<int32_t>(v.Cp);
  a.tiles_m = static_cast<int32_t>((d + 127) / 128);
  p.sn = static_cast<uint32_t>(v.Hp * v.Wp * px); p.sy = static_cast<uint32_t>(sh * v.Wp * px); p.sx = static_cast<uint32_t>(sw * px);
  p.M = static_cast<int32_t>(M); p.Ho = static_cast<int32_t>(v.Ho); p.Wo = static_cast<int32_t>(v.Wo);
  p.mWo = make_magic(p.Wo); p.mHo = make_magic(p.Ho);
  p.ntaps = static_cast<int32_t>(KK); p.kw = kw; p.pitch = static_cast<uint32_t>(v.Wp * px);
  p.tiles_n = a.tiles_m;
  // as few rounds of stages as the device takes, an item 13 of its own and the partial tiles one per 20 (corr3_plan_build)
  const int64_t tiles = static_cast<int64_t>(a.tiles_m) * (a.tiles_m + 1) / 2, all = (M + kC3K - 1) / kC3K;
  int64_t best = 1;
  double best_time = 0;
  for (int64_t ns = 1; ns <= std::max<int64_t>(1, std::min<int64_t>(all / 4, 512 / tiles + 1)); ++ns) {
    const double time = static_cast<double>((tiles * ns + 255) / 256 * ((all + ns - 1) / ns + 13)) + 0.05 * static_cast<double>(tiles * ns);
    if (ns == 1 || time < best_time) best = ns, best_time = time;
  }
  p.k_split = static_cast<int32_t>(((all + best - 1) / best + 1) / 2 * 2);
  p.nsplit = static_cast<int32_t>((all + p.k_split - 1) / p.k_split);
  v.items = static_cast<int>(tiles * p.nsplit);
  v.part_at = (static_cast<size_t>(v.plane_bytes) + 255) & ~static_cast<size_t>(255);
  v.ws_bytes = v.part_at + static_cast<size_t>(v.items) * 65536;
  return true;
}

// Against the fp32 kernel of syrk_window.hpp, which multiplies 64 x 64 tiles at 46 to 82 TFLOP/s: here 18 us for three launches, 3.5 TB/s
// into the planes, 0.45 us per stage of a round of 128 x 128 tiles (13 of a tile's own; a sixth of the matrix cores' bf16 rate), the
// latency of the splits' sum, and the partial tiles, 64 KB that are written and read again at 5 TB/s, also of a single split.  The last is what
// factors of many columns and few positions spend their time on (2 x 1600 x 9 x 9, 3 x 3 / 2, 50 positions: 434 us there, 555 here).
// us there and here: samples x channels x image, 3 x 3 / 2: 128 x 64 x 32 x 32 231 and 115, 32 x 64 x 32 x 32 72 and 48,
// 8 x 64 x 32 x 32 28 and 34, 128 x 96 x 8 x 8 38 and 37, 128 x 192 x 4 x 4 34 and 36, 32 x 300 x 14 x 14 188 and 125, 64 x 1024 x 4 x 4 354 and 301,
// 16 x 1024 x 4 x 4 173 and 243, 16 x 2048 x 4 x 4 778 and 891, 64 x 2048 x 4 x 4 1410 and 1137; 3 x 3 / 1: 128 x 32 x 32 x 32 270 and 162,
// 128 x 32 x 16 x 16 72 and 74, 128 x 20 x 32 x 32 140 and 157, 128 x 24 x 32 x 32 183 and 157, 128 x 96 x 16 x 16 391 and 163,
// 8 x 300 x 7 x 7 60 and 64; 5 x 5 of 16 x 24 x 56 x 56 295 and 214; 2 x 2 / 2 of 128 x 64 x 16 x 16 34 and 60.  Over 90 windows of 24 to 2048 channels the
// choice is 0.6 % from the faster one on average, at worst 53 us for 41 (5 x 189 x 14 x 14, 3 x 3 / 1 without padding).  The partial tiles take
// half the factor's own bytes and 34 MB at most (more than one split only below 512 tiles).
static bool corr3_window_faster(const Corr3Window& v, int64_t C, int kh, int kw) {
  const Corr3Prod& p = v.args.prod[0];
  const double T = static_cast<double>((C * kh * kw + 63) / 64), rounds = (v.items + 255) / 256;
  const double there = T * (T + 1) / 2 * 8192 * p.M / 55e6;
  const double here = 18 + static_cast<double>(v.plane_bytes) / 3.5e6 + 0.45 * rounds * (p.k_split + 13) + 0.3 * p.nsplit + v.items * 131072.0 / 5e6;
  return here < there;
}

size_t conv_window_f32_ws_bytes(int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int ph, int pw) {
  Corr3Window v;
  return corr3_window_plan(v, N, C, H, W, kh, kw, sh, sw, ph, pw) && corr3_window_faster(v, C, kh, kw) ? v.ws_bytes : 0;
}

int conv_window_syrk_f32(const float* x, int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int ph, int pw, float alpha,
                         float beta, float* A, int64_t lda, void* ws, size_t ws_bytes, hipStream_t stream) {
  Corr3Window v;
  if (!corr3_window_plan(v, N, C, H, W, kh, kw, sh, sw, ph, pw) || !corr3_window_faster(v, C, kh, kw)) return AK_ERR_UNSUPPORTED;
  if (ws == nullptr || ws_bytes < v.ws_bytes || (reinterpret_cast<uintptr_t>(ws) & 255) != 0) return AK_ERR_WORKSPACE;
  constexpr int kLds = kC3Stages * 4 * 6 * 1024;
  static bool attr_set = false;     // idempotent; a race sets it twice at worst
  if (!attr_set) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(corr3_products_kernel<2, 2, true>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
      return AK_ERR_LAUNCH;
    attr_set = true;
  }
  unsigned char* base = static_cast<unsigned char*>(ws);
  const int KK = kh * kw;
  v.args.planes = base;
  v.args.part = reinterpret_cast<floatx4*>(base + v.part_at);
  hipLaunchKernelGGL(corr3_split_kernel, dim3(static_cast<unsigned>((v.Hp * v.Wp + 31) / 32), static_cast<unsigned>(v.Cp / 32), static_cast<unsigned>(N)),
                     dim3(256), 0, stream, x, reinterpret_cast<uint16_t*>(base), static_cast<int>(C), static_cast<int>(v.Cp), static_cast<int>(H),
                     static_cast<int>(W), static_cast<int>(v.Hp), static_cast<int>(v.Wp), ph, pw);
  hipLaunchKernelGGL((corr3_products_kernel<2, 2, true>), dim3(static_cast<unsigned>(v.items)), dim3(256), kLds, stream, v.args);
  hipLaunchKernelGGL(corr3_window_kernel, dim3(static_cast<unsigned>(v.Cp / 32), static_cast<unsigned>((C + 7) / 8), static_cast<unsigned>(KK)), dim3(v.args.prod[0].nsplit > 8 ? 64 * std::min(KK, 16) : 256),
                     8 * (32 * KK + 1) * sizeof(float), stream, v.args, KK, static_cast<int>(C), alpha, beta, A, lda);
  return check_launch();
}

}  // namespace ak
