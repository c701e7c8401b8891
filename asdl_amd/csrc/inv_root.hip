// Shampoo's inverse p-th roots of symmetric PSD statistics, in groups of one size n and power p each:
//   out <- (S + r I)^(-1/p),  r = ridge_eps * lambda_max(S),
// lambda_max by the power iteration of the reference, then a coupled Newton iteration, every convergence test
// evaluated on the device: each kernel reads its matrix's `active` word first and returns at once when that matrix has
// converged (or stopped because its error grew, in which case the previous root is kept).
//
// Power iteration.  The estimate after k steps is mu_{2k+1} / mu_{2k} with mu_j = v0^T S^j v0, a functional of the spectral
// measure of v0.  32 Lanczos steps give the tridiagonal matrix T whose measure matches it (the first 63 moments exactly,
// and what dominates the higher ones, the top of the spectrum, to rounding); the power iteration itself, with its stopping
// rule and its limit of 100 steps, then runs on T in the registers of one wave.  Same estimate to 1e-6 (fp32 rounding),
// a third of the passes over the statistics and a sixth of the launches.
//
// Newton iteration.  M_0 = z S, X_0 = z^(1/p) I;  T = a I - b M;  X <- X T;  M <- T^p M.  The classical step a = 1 + 1/p,
// b = 1/p raises a small eigenvalue of M by (1 + 1/p)^p = 2.44 (p = 4): most of its 20 steps on a statistic of condition 1e6.
// With a lower bound l of the spectrum known (from the Lanczos steps, at the least the ridge) the step that raises l most is a
// larger a with b = a^(p+1) p^p / (p+1)^(p+1), which keeps max m (a - b m)^p = 1: up to 7.4 per step.  root_schedule_kernel
// decides per matrix whether that is the shorter way.
// For p = 4 T is a polynomial of the fourth degree there: two products more than a classical step's four, P = 2 U^2 - I with
// U = 2 M - I and T = t(U, P) + P y(U, P), for a factor of 29 per step where the first degree, held to the same top of the
// spectrum, has 4.6: 10 or 11 steps and 45 to 51 products where 15 or 16 steps of the first degree took 59 to 63 (98 statistics of
// 768 to 3072 columns 140 -> 122 ms, 111 without the last step's M' (root_settled_kernel); the device's power limit holds the products of
// all of them near 1.15 PFLOP/s of fp16).
// Its rounding: T^4 reaches 29, and T^4 M inherits what rounding T^4 does, that much larger than the top of the spectrum it is
// added to.  Behind the early steps M' is therefore (T^2 M) T^2, and T^2 and X T are formed from D = T - I as D^2 + 2 D + I
// and X D + X: without either the root lost a factor of 3.5 where the gradient lies, with both it gains (root_schedule_kernel).
// The first kRootEarly steps stay classical, in the summation order of one fixed kernel per size.  What an ill-conditioned
// root ends up with is decided there: the rounding of M' perturbs the smallest eigenvalues by about 5e-8, 1 to 2 % of the
// root at condition 1e6, and every later step's perturbation counts 2.44 times less.  Another order, though as accurate, gives
// another root within that percent; rank-deficient statistics of 625 to 1498 columns differ from the root of the wholly
// classical iteration by 0.6 to 0.9 % after three classical steps, by 0.12 to 0.17 % after five (one step more).
//
// The matrices of the iteration, all polynomials of one symmetric matrix, are kept
//  * as 16-bit planes from 512 columns up (gemm_planes.hpp), of which only tiles on one side of the diagonal are computed,
//    and mirrored: 192 x 192 tiles, one launch per product and group, where a group
//    has enough of them to fill the device, else 64 x 64 tiles;
//  * in fp32 below, every tile of a product computed: with mirrored tiles the part of the rounding that is not symmetric
//    goes elsewhere, and the root of a rank-deficient statistic moves by most of its own error (1 % at 255 columns).
// The small tiles of all groups of a kind share one launch per step of the product sequence.
// All sum in chunks; the product that forms the next M also folds max |M - I| into a device word and writes the next
// step's polynomial T.  X, M and T alternate between two buffers by the parity of the matrix's own step count: nothing is
// copied per step and a rejected step leaves its matrix where it was.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include "gemm_f32.hpp"
#include "gemm_planes.hpp"

namespace ak {

constexpr int RCHUNKS = 64;             // partial-reduction chunks per matrix
constexpr int kRootMaxGroups = 16;      // groups of one call (they travel in the kernel arguments)
constexpr int kLanczosSteps = 32;
constexpr int kLanczosLdsDim = 32768;  // columns whose vector is kept in the LDS (128 of its 160 KB)
constexpr int kLanczosRows = 16;        // rows of the statistic per work group and step: four waves, four rows each
constexpr int kRootEarly = 5;           // classical steps before the accelerated ones
constexpr int kRootSteps = 32;          // entries of a matrix's step table; the last one repeats
constexpr int kRootFixedBuffers = 6;    // R0 R1 M0 M1 T0 T1; product buffers behind them (root_buffers)
constexpr int kRootMinPlaneDim = 512;

// Scales of the two-plane fp16 form (gemm_planes.hpp).  M and the polynomials are bounded by the normalisation of the iteration:
// M <= (1 + p) / 2; T^p of a step of the first degree is at most 12 (root_schedule_kernel); of a step of the fourth degree T^2 is at
// most 5.5 and T^4 29, which is never stored: M' is (T^2 M) T^2 there (root_ops).  So 2^12 keeps them (and a fair excess of an
// indefinite input) below the fp16 maximum.  The root is kept without its factor z^(1/p): it grows from I to
// (z A)^(-1/p) <= lambda_min(M_0)^(-1/p), and the ridge bounds lambda_min(M_0) >= ridge_eps (1 + p) / (2 sqrt(n)) from
// below (lambda_max from the power iteration; a value that is low by a factor f moves the bound by f^(1/p), which the four
// spare bits cover).  The root's scale must
// not be below one (the identity it starts from needs its 22 bits too), so the bound has to stay below 2^12: p = 4 with a
// ridge of 1e-6 gives 70, p = 2 at the same ridge 8000 and more.  Beyond that, without a ridge, or with a power above 8
// the iteration stays on the bf16 planes, which have the range of fp32.
constexpr float kRootScaleM = 4096.f;
static bool root_fp16_allowed() {
  static const bool on = [] {
    const char* e = std::getenv("ASDL_AMD_ROOT_FP16_PLANES");
    return e == nullptr || e[0] != '0';
  }();
  return on;
}
static bool root_plane_dim(int64_t n) { return n >= kRootMinPlaneDim && n <= kPlaneMaxDim; }
// 0: not on fp16 planes; else the scale of the root's planes
static float root_fp16_scale(int64_t n, int p, float ridge_eps) {
  if (!root_fp16_allowed() || !root_plane_dim(n) || p > 8 || !(ridge_eps > 0.f)) return 0.f;
  const double lam = static_cast<double>(ridge_eps) * (1 + p) / (2.0 * std::sqrt(static_cast<double>(n)));
  const double bound = std::pow(lam, -1.0 / p);                 // of the root's largest eigenvalue
  if (!(bound < 1e30)) return 0.f;
  const int e = 12 - static_cast<int>(std::ceil(std::log2(bound)));
  if (e < 0) return 0.f;
  return static_cast<float>(std::ldexp(1.0, e < 12 ? e : 12));
}
static int64_t root_pad(int64_t n, int tile) { return (n + tile - 1) / tile * tile; }
static int64_t root_ld(int64_t n) { return (n + 3) / 4 * 4; }

// Tile of a group on planes.  A 192-wide tile takes 0.75 us per k-tile of 16 and CU however few there are; a 64-wide one
// 0.55 us per 64 k beside 5 us of latency for every 256 of them (1024 columns 14.5 us a product, 1536 28, where the wide tile takes 72).
static int root_plane_tile(int64_t n, int64_t batch) {
  const double big = static_cast<double>(root_pad(n, kPlaneTile)), small = static_cast<double>(root_pad(n, kPlaneSmallTile));
  const double T = big / kPlaneTile, t = small / kPlaneSmallTile;
  const double us_big = std::max(1.0, T * (T + 1) / 2 * batch / 256) * (big / 16) * 0.75;
  const double us_small = std::ceil(t * (t + 1) / 2 * batch / 256) * (5.0 + small / 64 * 0.55);
  return us_small < us_big ? kPlaneSmallTile : kPlaneTile;
}

// Storage of the matrices of a group: 0 (fp32), 2 or 3 planes.
static int root_planes(int64_t n, int p, float ridge_eps) {
  return !root_plane_dim(n) ? 0 : (root_fp16_scale(n, p, ridge_eps) > 0.f ? 2 : 3);
}

// fp32 groups with many wide matrices take 128 x 128 tiles.
static bool root_split(int64_t n, int64_t batch) {
  const int64_t t = (n + 127) / 128;
  return t * t * batch >= 100 && n >= 256 && n % 4 == 0;
}

// floats of one matrix buffer of a statistic
static size_t root_buffer_floats(int64_t n, int64_t batch, int np) {
  if (np == 0) return static_cast<size_t>(n) * root_ld(n);
  const size_t n_pad = static_cast<size_t>(root_pad(n, root_plane_tile(n, batch)));
  return np * n_pad * n_pad / 2;
}

struct RootState {
  // per matrix of the call, all device memory
  float* sv;        // eigenvalue estimate
  float* err;       // Newton error max|M - I| of the accepted steps
  float* zscale;
  float* partial;   // [RCHUNKS]: sums of squares, then max |M_0 - I|
  float* alpha;     // [kLanczosSteps] the tridiagonal matrix: diagonal,
  float* beta;      // [kLanczosSteps] and beta[j] next to alpha[j - 1], alpha[j]
  float* coef;      // [kRootSteps kCoefs]: a, b and the quartic's coefficients of every step (gemm_planes.hpp)
  float* errword;   // [kErrSlots kErrStride] max |M' - I| of the step under way, folded in by the epilogue of the product that forms M'
  int* lz_dim;      // Lanczos steps that counted (0: all)
  int* pi_iters;
  int* active;      // Newton iteration still running
  int* count;       // accepted steps
  int* accel;       // steps of the table that are not the classical one
  int* ovf;         // fp16 planes: a product of the step under way left the fp16 range
  float* settled;   // > 0: the next step is the last one and needs no M' (root_settled_kernel); what bounds its error
  // err, active, count, ovf and errword have a second half, `total` entries further on: root_small_kernel
  int total;
};

struct RootGroup {
  float* S;
  float* out;
  const float* v0;
  float* stats;
  float* bufs;          // `buffers` buffers of `batch` fp32 matrices (n rows of ld) or plane sets
  float* vec;           // Lanczos vectors: q ring of 3, S q ring of 2, each [batch, n]
  int64_t strideS, strideOut;
  int n, ld, batch, p, buffers;
  int z0;               // first matrix of the group in the state arrays
  int np, n_pad, tile;  // planes per matrix: 0 (fp32), 2, 3; tile of the products on planes
  int quartic;          // steps of the fourth degree are among its products
  float scale_r;
};
struct RootGroups {
  RootState st;
  int count, total;
  RootGroup g[kRootMaxGroups];
};

// Entry z (total + z: of the second half) of what the products of a step fold into.
__device__ __forceinline__ void root_clear_words(const RootState& st, int z) {
  for (int s = 0; s < kErrSlots; ++s) st.errword[(z * kErrSlots + s) * kErrStride] = 0.f;
  st.ovf[z] = 0;
}

__device__ __forceinline__ int root_group_of(const RootGroups& G, int z) {
  int g = 0;
  while (g + 1 < G.count && G.g[g + 1].z0 <= z) ++g;
  return g;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}
// Sum over the 256 threads of a work group, the same value in all of them.  red: 4 floats, free again after the next barrier.
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// What a Lanczos step needs of a group; `first`: its first work group.  (The first numbers of all groups lie side by side: a
// work group finds its own with one load.  Kernel arguments behind a dependent index cost a trip to memory each.)
struct LanczosGroup {
  const float* S;
  const float* v0;
  float* vec;
  float* parts;
  int64_t strideS;
  int n, batch, z0, pad;
};
struct LanczosGroups {
  int first[kRootMaxGroups];
  LanczosGroup g[kRootMaxGroups];
};

// Lanczos step j: q_j from S q_{j-1}, then its work group's rows of S q_j.  Every work group of a matrix forms q_j for
// itself in the LDS (three vectors from the L2, two reductions): one launch per step, no hand-over inside it.  The
// rows of S are requested before that, their first 1024 columns kept in registers.
// Bound by the launch and the chain of loads and reductions; where it would be by reading S, root_lanczos_tiles_kernel reads half.
// WIDE: vectors that the LDS does not hold (kLanczosLdsDim) are formed again, element by element, where they are used.
// HELD: at most 1024 columns, and work groups that wait rather than fill the memory: the three vectors come into registers and are
// requested first (loads return in order), then the rows of S, none under a lane's own condition, which would be waited for by
// itself.  784 and 512 columns: 7.4 -> 6.0 us a step; 98 matrices of up to 3072 columns, bound by reading S, lose 7 % by it.
template <bool WIDE, bool HELD>
static __global__ __launch_bounds__(256) void root_lanczos_kernel(RootState st, LanczosGroups L, int j) {
  extern __shared__ __attribute__((aligned(16))) float q[];
  __shared__ float red[3][4];
  const int wg = blockIdx.x;
  int gi = 0;
#pragma unroll
  for (int k = 1; k < kRootMaxGroups; ++k) gi += wg >= L.first[k] ? 1 : 0;
  const LanczosGroup g = L.g[gi];
  const int n = g.n, per = (n + kLanczosRows - 1) / kLanczosRows;
  const int local = wg - L.first[gi], zl = local / per, part = local - zl * per;
  const int z = g.z0 + zl, tid = threadIdx.x, lane = tid & 63, row0 = part * kLanczosRows + 4 * (tid >> 6);
  const float* __restrict__ S = g.S + zl * g.strideS;
  const int n4 = n & ~3;
  const int64_t vec = static_cast<int64_t>(g.batch) * n;
  float* __restrict__ qj = g.vec + (j % 3) * vec + static_cast<int64_t>(zl) * n;
  const float* __restrict__ v0 = g.v0 + static_cast<int64_t>(zl) * n;
  const float* __restrict__ q1 = g.vec + ((j + 2) % 3) * vec + static_cast<int64_t>(zl) * n;
  const float* __restrict__ q2 = g.vec + ((j + 1) % 3) * vec + static_cast<int64_t>(zl) * n;
  const float* __restrict__ w = g.vec + (3 + ((j + 1) & 1)) * vec + static_cast<int64_t>(zl) * n;
  float hw[4], h1[4], h2[4];
  floatx4 early[4][4];
  if constexpr (HELD) {
    const float* __restrict__ first = j == 0 ? v0 : w;
#pragma unroll
    for (int u = 0; u < 4; ++u) {      // (elements beyond the end read the last one and are not used)
      const int i = min(tid + 256 * u, n - 1);
      hw[u] = first[i];
      h1[u] = q1[i];
      h2[u] = q2[i];
    }
    if (n4 > 0) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int k = min(4 * lane + 256 * c, n4 - 4), row = row0 + r < n ? row0 + r : n - 1;
          early[c][r] = *reinterpret_cast<const floatx4u*>(S + static_cast<int64_t>(row) * n + k);
        }
    }
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 4 * lane + 256 * c, row = row0 + r < n ? row0 + r : n - 1;
        early[c][r] = k < n4 ? *reinterpret_cast<const floatx4u*>(S + static_cast<int64_t>(row) * n + k) : floatx4{0.f, 0.f, 0.f, 0.f};
      }
  }
  float a = 0.f, b = 0.f, inv = 0.f;
  auto raw = [&](int i) { return j == 0 ? v0[i] : w[i] - a * q1[i] - (j > 1 ? b * q2[i] : 0.f); };     // q_j without its scale
  auto form = [&](float* sums) {                      // the vector (WIDE: nothing) and its length
    float s = 0.f;
    if constexpr (HELD) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = tid + 256 * u;
        if (i >= n) break;
        const float x = j == 0 ? hw[u] : hw[u] - a * h1[u] - (j > 1 ? b * h2[u] : 0.f);
        q[i] = x;
        s += x * x;
      }
    } else {
      for (int i = tid; i < n; i += 256) {
        const float x = raw(i);
        if constexpr (!WIDE) q[i] = x;
        s += x * x;
      }
    }
    return sqrtf(block_sum(s, sums));
  };
  auto scale = [&] {
    for (int i = tid; i < n; i += 256) {
      if constexpr (!WIDE) q[i] *= inv;
      if (part == 0) {
        if constexpr (WIDE) qj[i] = raw(i) * inv;
        else qj[i] = q[i];
      }
    }
  };
  if (j == 0) {
    inv = 1.f / form(red[0]);
    scale();
    if (part == 0 && tid == 0) {
      st.lz_dim[z] = 0;
      st.active[z] = st.count[z] = 0;
      st.settled[z] = 0.f;
      root_clear_words(st, z);
      root_clear_words(st, st.total + z);
      st.beta[z * kLanczosSteps] = 0.f;
    }
  } else {
    if (j > 1 && st.lz_dim[z] != 0) return;            // an invariant subspace: T is complete
    b = st.beta[z * kLanczosSteps + j - 1];
    float s = 0.f;
    if constexpr (HELD) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (tid + 256 * u < n) s += hw[u] * h1[u];
    } else {
      for (int i = tid; i < n; i += 256) s += w[i] * q1[i];
    }
    a = block_sum(s, red[0]);
    const float norm = form(red[1]);
    const bool done = !(norm > 1e-7f * fabsf(a));
    if (part == 0 && tid == 0) {
      st.alpha[z * kLanczosSteps + j - 1] = a;
      if (done) st.lz_dim[z] = j;
      else st.beta[z * kLanczosSteps + j] = norm;
    }
    if (done) return;
    inv = 1.f / norm;
    scale();
  }
  __syncthreads();
  auto four = [&](int k) {
    if constexpr (!WIDE) return *reinterpret_cast<const floatx4*>(q + k);
    else return floatx4{raw(k), raw(k + 1), raw(k + 2), raw(k + 3)} * inv;
  };
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int k = 4 * lane + 256 * c;
    if (k >= n4) break;
    const floatx4 x = four(k);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      acc[r] += early[c][r][0] * x[0] + early[c][r][1] * x[1] + early[c][r][2] * x[2] + early[c][r][3] * x[3];
  }
  for (int k = 4 * lane + 1024; k < n4; k += 256) {
    const floatx4 x = four(k);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + r < n ? row0 + r : n - 1;
      const floatx4 m = *reinterpret_cast<const floatx4u*>(S + static_cast<int64_t>(row) * n + k);
      acc[r] += m[0] * x[0] + m[1] * x[1] + m[2] * x[2] + m[3] * x[3];
    }
  }
  if (n4 + lane < n) {
    float x;
    if constexpr (WIDE) x = raw(n4 + lane) * inv;
    else x = q[n4 + lane];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + r < n ? row0 + r : n - 1;
      acc[r] += S[static_cast<int64_t>(row) * n + n4 + lane] * x;
    }
  }
  float* __restrict__ wj = g.vec + (3 + (j & 1)) * vec + static_cast<int64_t>(zl) * n;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float s = wave_sum(acc[r]);
    if (lane == 0 && row0 + r < n) wj[row0 + r] = s;
  }
}

// Lanczos steps of many large statistics, bound by reading S: its lower triangle alone, by tiles of 256 x 256 that serve both sides, and
// the sum of their parts and the vectors in a launch between, a work group per matrix.  98 matrices of up to 3072 columns (1.3 GB):
// a step 229 us, now 135 (8 rows' loads at a time instead of 16: 144) and 13.  From which sum of bytes on: the whole roots cut off after
// one step, by whole rows and by halves, 3 x 3072 (113 MB) 2.24 and 2.32 ms, 5 x 3072 3.22 and 3.10, 11 x 3072 6.82 and 5.61;
// 40 x 768 (94 MB) 1.32 and 1.35, 80 x 768 2.24 and 1.96.
constexpr int kLanczosTile = 256;
constexpr int64_t kLanczosHalfBytes = 128ll << 20;
// (from 64 columns on a matrix's buffers hold its parts)
static bool lanczos_halves(int64_t widest, int64_t narrowest, int64_t bytes) {
  return widest <= kLanczosLdsDim && narrowest >= 64 && bytes >= kLanczosHalfBytes;
}
// parts: [batch][block of rows][block of columns][256], in the matrix buffers, which nothing else uses yet
__device__ __forceinline__ float* lanczos_parts(float* bufs, int nb, int zl) { return bufs + static_cast<int64_t>(zl) * nb * nb * kLanczosTile; }

// The parts of S q_j.
static __global__ __launch_bounds__(256) void root_lanczos_tiles_kernel(RootState st, LanczosGroups L, int j) {
  constexpr int ROWS = 16, LANES = 64 / ROWS;
  __shared__ floatx4 sums[4][64];
  const int wg = blockIdx.x;
  int gi = 0;
#pragma unroll
  for (int k = 1; k < kRootMaxGroups; ++k) gi += wg >= L.first[k] ? 1 : 0;
  const LanczosGroup g = L.g[gi];
  const int n = g.n, nb = (n + kLanczosTile - 1) / kLanczosTile, per = nb * (nb + 1) / 2;
  const int local = wg - L.first[gi], zl = local / per, t = local - zl * per;
  if (j > 0 && st.lz_dim[g.z0 + zl] != 0) return;
  int bi, bj;
  decode_lower_tile(t, bi, bj);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, row0 = kLanczosTile * bi + 64 * wave, col = kLanczosTile * bj + 4 * lane;
  const float* __restrict__ S = g.S + zl * g.strideS;
  const float* __restrict__ q = g.vec + (j % 3) * (static_cast<int64_t>(g.batch) * n) + static_cast<int64_t>(zl) * n;
  float* __restrict__ parts = lanczos_parts(g.parts, nb, zl);
  const bool whole = kLanczosTile * (bj + 1) <= n;         // (the last tile of the diagonal may reach beyond the matrix)
  floatx4 x = {0.f, 0.f, 0.f, 0.f}, down = x;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (col + e < n) x[e] = q[col + e];
  const float mine = row0 + lane < n ? q[row0 + lane] : 0.f;
  auto sweep = [&](auto whole_tag) {
    for (int r0 = 0; r0 < 64; r0 += ROWS) {
      floatx4 m[ROWS];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {                     // (rows beyond the end read the last one, times zero)
        const float* __restrict__ src = S + static_cast<int64_t>(min(row0 + r0 + r, n - 1)) * n;
        if constexpr (decltype(whole_tag)::value) m[r] = *reinterpret_cast<const floatx4u*>(src + col);
        else
#pragma unroll
          for (int e = 0; e < 4; ++e) m[r][e] = src[min(col + e, n - 1)];
      }
      float v[ROWS];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const float y = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine), r0 + r));
        v[r] = m[r][0] * x[0] + m[r][1] * x[1] + m[r][2] * x[2] + m[r][3] * x[3];
        down += m[r] * y;
      }
      // the rows' sums over the lanes, half as many with every exchange: lanes LANES r ... end with row r's
#pragma unroll
      for (int o = 32, h = ROWS / 2; h >= 1; o >>= 1, h >>= 1)
#pragma unroll
        for (int r = 0; r < h; ++r) {
          const bool up = (lane & o) != 0;
          v[r] = (up ? v[r + h] : v[r]) + __shfl_xor(up ? v[r] : v[r + h], o);
        }
#pragma unroll
      for (int o = LANES / 2; o >= 1; o >>= 1) v[0] += __shfl_xor(v[0], o);
      if (lane % LANES == 0) parts[static_cast<int64_t>(bi * nb + bj) * kLanczosTile + 64 * wave + r0 + lane / LANES] = v[0];
    }
  };
  if (whole) sweep(std::true_type{});
  else sweep(std::false_type{});
  if (bi == bj) return;
  sums[wave][lane] = down;
  __syncthreads();
  const float* all = reinterpret_cast<const float*>(sums);
  parts[static_cast<int64_t>(bj * nb + bi) * kLanczosTile + tid] = (all[tid] + all[256 + tid]) + (all[512 + tid] + all[768 + tid]);
}

// Sum over the 1024 threads of a work group; red: 16 floats of this sum's own.
__device__ __forceinline__ float block_sum_1024(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < 16; ++k) s += red[k];
  return s;
}

// S q_{j-1} from its parts, T's entries and q_j (root_lanczos_kernel's); j = steps: S q_{j-1} alone, for T's last entry.  grid (total).
static __global__ __launch_bounds__(1024) void root_lanczos_vector_kernel(RootState st, LanczosGroups L, int j, int steps) {
  __shared__ float red[2][16];
  const int z = blockIdx.x, tid = threadIdx.x;
  int gi = 0;
#pragma unroll
  for (int k = 1; k < kRootMaxGroups; ++k) gi += L.first[k] != INT32_MAX && z >= L.g[k].z0 ? 1 : 0;
  const LanczosGroup g = L.g[gi];
  const int n = g.n, nb = (n + kLanczosTile - 1) / kLanczosTile, zl = z - g.z0;
  const int64_t vec = static_cast<int64_t>(g.batch) * n, at = static_cast<int64_t>(zl) * n;
  float* __restrict__ qj = g.vec + (j % 3) * vec + at;
  if (j == 0) {
    const float* __restrict__ v0 = g.v0 + at;
    float s = 0.f;
    for (int i = tid; i < n; i += 1024) s += v0[i] * v0[i];
    const float inv = 1.f / sqrtf(block_sum_1024(s, red[0]));
    for (int i = tid; i < n; i += 1024) qj[i] = v0[i] * inv;
    if (tid == 0) {
      st.lz_dim[z] = 0;
      st.active[z] = st.count[z] = 0;
      st.settled[z] = 0.f;
      root_clear_words(st, z);
      root_clear_words(st, st.total + z);
      st.beta[z * kLanczosSteps] = 0.f;
    }
    return;
  }
  if (st.lz_dim[z] != 0) return;
  const float* __restrict__ q1 = g.vec + ((j + 2) % 3) * vec + at;
  const float* __restrict__ q2 = g.vec + ((j + 1) % 3) * vec + at;
  float* __restrict__ w = g.vec + (3 + ((j + 1) & 1)) * vec + at;
  const float* __restrict__ parts = lanczos_parts(g.parts, nb, zl);
  const float b = st.beta[z * kLanczosSteps + j - 1];
  float s = 0.f;
  for (int i = tid; i < n; i += 1024) {
    const float* __restrict__ src = parts + static_cast<int64_t>(i / kLanczosTile) * nb * kLanczosTile + i % kLanczosTile;
    float x = 0.f;
#pragma unroll 4
    for (int c = 0; c < nb; ++c) x += src[c * kLanczosTile];
    w[i] = x;
    s += x * q1[i];
  }
  if (j == steps) return;
  const float a = block_sum_1024(s, red[0]);
  s = 0.f;
  for (int i = tid; i < n; i += 1024) {                    // (a thread's own elements of w)
    const float x = w[i] - a * q1[i] - (j > 1 ? b * q2[i] : 0.f);
    w[i] = x;
    s += x * x;
  }
  const float norm = sqrtf(block_sum_1024(s, red[1]));
  const bool done = !(norm > 1e-7f * fabsf(a));
  if (tid == 0) {
    st.alpha[z * kLanczosSteps + j - 1] = a;
    if (done) st.lz_dim[z] = j;
    else st.beta[z * kLanczosSteps + j] = norm;
  }
  if (done) return;
  const float inv = 1.f / norm;
  for (int i = tid; i < n; i += 1024) qj[i] = w[i] * inv;
}

template <int CTRL>
__device__ __forceinline__ float dpp_zero(float v) {       // lanes without a source read zero
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// Sum over lanes 0 ... 31, the same value everywhere.
__device__ __forceinline__ float sum32(float v) {
  v += dpp_zero<0x111>(v);       // row_shr:1, 2, 4, 8: lane 15 of a row of 16 holds its sum
  v += dpp_zero<0x112>(v);
  v += dpp_zero<0x114>(v);
  v += dpp_zero<0x118>(v);
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 15)) +
         __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 31));
}

// grid (total), one wave: the reference's power iteration (estimate (v/|v|) . S v/|v|, stop on |change| <= tol) on T.
static __global__ __launch_bounds__(64) void root_power_kernel(RootGroups G, int steps, float tol, int max_iters) {
  const int z = blockIdx.x, lane = threadIdx.x;
  const RootGroup& g = G.g[root_group_of(G, z)];
  const int zl = z - g.z0;
  int m = G.st.lz_dim[z];
  if (m == 0) {
    // the last diagonal element: q . S q of the last step
    const int64_t vec = static_cast<int64_t>(g.batch) * g.n, at = static_cast<int64_t>(zl) * g.n;
    const float* __restrict__ q = g.vec + ((steps - 1) % 3) * vec + at;
    const float* __restrict__ w = g.vec + (3 + ((steps - 1) & 1)) * vec + at;
    float s = 0.f;
    for (int i = lane; i < g.n; i += 64) s += q[i] * w[i];
    s = wave_sum(s);
    if (lane == 0) G.st.alpha[z * kLanczosSteps + steps - 1] = s;
    m = steps;
    __syncthreads();
  }
  float a = 0.f, bl = 0.f, br = 0.f;           // diagonal, couplings to the lanes below and above
  if (lane < m) {
    a = G.st.alpha[z * kLanczosSteps + lane];
    if (lane > 0) bl = G.st.beta[z * kLanczosSteps + lane];
    if (lane + 1 < m) br = G.st.beta[z * kLanczosSteps + lane + 1];
  }
  float v = lane == 0 ? 1.f : 0.f, sv = 0.f;
  int it = 0;
  bool go_on = max_iters > 0;
  while (go_on) {
    const float x = v / sqrtf(sum32(v * v));
    const float y = a * x + bl * dpp_zero<0x138>(x) + br * dpp_zero<0x130>(x);      // wave_shr:1, wave_shl:1
    const float s = sum32(x * y);
    const float error = fabsf(s - sv);
    sv = s;
    v = y;
    ++it;
    go_on = error > tol && it < max_iters;
  }
  if (lane == 0) {
    G.st.sv[z] = sv;
    G.st.pi_iters[z] = it;
  }
}

// grid (RCHUNKS, total): S += ridge I (in place), partial sum of squares of the ridged matrix
static __global__ __launch_bounds__(256) void root_ridge_kernel(RootGroups G, float ridge_eps) {
  __shared__ float red[4];
  const int z = blockIdx.y;
  const RootGroup& g = G.g[root_group_of(G, z)];
  float* __restrict__ S = g.S + (z - g.z0) * g.strideS;
  const float ridge = ridge_eps * G.st.sv[z];
  const uint32_t total = static_cast<uint32_t>(g.n) * static_cast<uint32_t>(g.n), period = static_cast<uint32_t>(g.n) + 1;
  float s = 0.f;
  if (g.n > kLanczosLdsDim) {                   // row by row: n^2 does not fit 32 bits
    for (int i = 4 * blockIdx.x + (threadIdx.x >> 6); i < g.n; i += 4 * RCHUNKS) {
      float* __restrict__ row = S + static_cast<int64_t>(i) * g.n;
      for (int k = threadIdx.x & 63; k < g.n; k += 64) {
        float x = row[k];
        if (k == i) row[k] = x += ridge;
        s += x * x;
      }
    }
  } else
#pragma unroll 4
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < total; i += RCHUNKS * 256) {
    float x = S[i];
    if (i % period == 0) {
      x += ridge;
      S[i] = x;
    }
    s += x * x;
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) G.st.partial[z * RCHUNKS + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

__device__ __forceinline__ float int_power(float x, int p) {
  float r = 1.f;
  for (int i = 0; i < p; ++i) r *= x;
  return r;
}

// Steps of the fourth degree (p = 4): T(m) = sum c_k T_k(2 m - 1), T_k the Chebyshev polynomials.  A row is for spectra in [l, 1],
// l its first entry, and raises their lower end most: max m T(m)^4 = 1, and where m T(m)^4 has left the rising edge at the
// lower end it stays at or above what it is at l (rows behind the first) or kRootQuarticTop (the first).  Solved as linear
// programmes on 3000 points: maximise v with v <= m^(1/4) T(m) on [l, 1] and m^(1/4) T(m) <= 1 on [0, 1].
constexpr float kRootQuarticTop = 0.85f;
constexpr int kRootQuarticRows = 13;
static __constant__ float kRootQuartics[kRootQuarticRows][6] = {
    {0.f, 1.36251366f, -0.54698689f, 0.24514824f, -0.11936991f, 0.05869484f},
    {0.075f, 1.35824512f, -0.52173189f, 0.22080282f, -0.09888875f, 0.04157265f},
    {0.1f, 1.35174999f, -0.49965946f, 0.20083153f, -0.08334540f, 0.03042332f},
    {0.13f, 1.34376311f, -0.47852429f, 0.18268849f, -0.07021425f, 0.02228694f},
    {0.17f, 1.33389297f, -0.45611605f, 0.16439933f, -0.05795065f, 0.01577439f},
    {0.22f, 1.32310502f, -0.43399607f, 0.14724395f, -0.04736485f, 0.01101190f},
    {0.28f, 1.31212364f, -0.41293058f, 0.13171368f, -0.03858015f, 0.00767336f},
    {0.36f, 1.29999203f, -0.39071790f, 0.11619157f, -0.03059383f, 0.00512813f},
    {0.45f, 1.28877730f, -0.37086123f, 0.10307336f, -0.02449238f, 0.00350292f},
    {0.55f, 1.27841119f, -0.35295083f, 0.09187384f, -0.01977349f, 0.00243930f},
    {0.65f, 1.26961606f, -0.33804700f, 0.08302710f, -0.01637640f, 0.00178024f},
    {0.75f, 1.26190359f, -0.32518863f, 0.07574798f, -0.01380495f, 0.00134192f},
    {0.85f, 1.25508714f, -0.31399054f, 0.06968431f, -0.01182153f, 0.00104061f},
};

// The smallest eigenvalue of T + ridge I (T: m Lanczos steps) within [lo, hi], from below and to 0.4 %; lo if it lies at or below
// that.  x lies below the spectrum where every pivot of T + (ridge - x) I is positive (Sturm): two rounds of 64 values of x, one per
// lane, in geometric progression.
__device__ __forceinline__ float lowest_ritz(const float* __restrict__ alpha, const float* __restrict__ beta, int m, float ridge,
                                             float lo, float hi) {
  const int lane = threadIdx.x;
#pragma unroll
  for (int round = 0; round < 2; ++round) {
    const float x = lo * powf(hi / lo, lane / 63.f);
    bool below = true;
    float d = 1.f;
    for (int i = 0; i < m; ++i) {
      const float c = i == 0 ? 0.f : beta[i];
      d = (alpha[i] + ridge - x) - c * c / d;
      below = below && d > 0.f;
    }
    const unsigned long long not_below = ~__ballot(below);
    if (not_below == 0) return hi;
    const int f = __ffsll(not_below) - 1;
    if (f == 0) return lo;
    hi = __shfl(x, f);
    lo = __shfl(x, f - 1);
  }
  return lo;
}

// Classical steps after which an eigenvalue m of M lies within tol of one, counted from step `from`.
__device__ __forceinline__ int classical_steps(float m, int p, float a0, float b0, float tol, int from) {
  int k = from;
  for (; k < 2 * kRootSteps && fabsf(m - 1.f) > tol; ++k) m *= int_power(a0 - b0 * m, p);
  return k;
}

// grid (total), one wave: the scale z and the (a, b) of every step.
//
// Two schedules are followed on the ends of the spectrum as the Lanczos steps saw it (the Ritz values of T, the ridge added), and the
// shorter one is used: the classical step throughout, or accelerated steps from a lower bound l of the spectrum.  l is half
// the smallest Ritz value, at least half the ridge's bound (the estimate of lambda_max may be low, S indefinite by its rounding).
// Too high a guess costs classical steps at the end, since eigenvalues below l rise faster than by the classical step too; too
// low a guess (the ridge's bound for a full-rank statistic) costs accelerated steps that nothing needs.  Steps at n = 512, p = 4, a ridge
// of 1e-6 (classical, from the ridge's bound throughout, by this rule): eigenvalues 1 ... 0.01 10, 15, 9; 1 ... 0.0001 15, 15, 13;
// summed batches of 128 rows, one (rank 128) 20, 15, 15, four 20, 15, 18, five 12, 15, 10, ten 9, 15, 8, forty 7, 15, 7.
// Accelerated steps also need a ridge of 1e-7 and more (below, the bound l is not one that fp32 can keep), a power up to 8, and room
// for the classical iteration's own number of steps (a caller that asks for a few steps gets those of the reference).
//
// A step may not press the top of the spectrum below kTopMin: its rounding error relative to that value is what the root inherits
// in the dominant directions, the ones that a gradient with this statistic lies in (the error of the whole root does not show
// it: that is the null space's, 1 to 2 % whatever the steps).  Error against fp64 of L^(-1/4) G R^(-1/4), L = G G^T, R = G^T G, and
// steps, for the classical iteration and kTopMin = 0.17, 0.5, 0.6, 0.7: G 512 x 784 of rank 128 5.6e-5 (20), 1.9e-4 (14), 8.3e-5 (15),
// 6.5e-5 (15), 5.1e-5 (15); 256 x 300, rank 64 6.6e-5 (20), 2.0e-4 (14), 7.8e-5 (14), 6.4e-5 (15), 5.8e-5 (15); 300 x 600, rank 16
// 1.2e-4 (20), 2.8e-4 (13), 1.5e-4 (14), 1.3e-4 (14), 1.3e-4 (15); 768 x 3072, rank 400 4.9e-5 (21), 1.3e-4 (14), 6.1e-5 (15),
// 5.4e-5 (15), 4.6e-5 (16).  0.7 is the first that loses nothing.  T^p of these steps stays below 12 for the fp16 planes.
// Steps of the fourth degree with the top at 0.7, 0.8, 0.85, 0.9 and, last, the first degree, on matrices of the first, second and fourth
// shape and 300 x 600 of rank 16: 5.7e-5 (10), 5.2e-5 (10), 4.9e-5 (10), 4.4e-5 (11), 5.2e-5 (15); 4.1e-5, 3.9e-5, 3.9e-5, 3.7e-5 (10 each), 5.9e-5 (15);
// 5.2e-5 (10), 4.8e-5 (10), 4.5e-5 (11), 4.2e-5 (11), 4.6e-5 (16); 6.5e-5, 6.2e-5, 6.0e-5, 6.0e-5 (10 each), 1.3e-4 (15).  0.85 is the lowest that
// loses nothing to speak of at any of 17 shapes from 64 x 50 to 2048 x 2048 (at the worst 3 %; on average it gains 15 %).
static __global__ __launch_bounds__(64) void root_schedule_kernel(RootGroups G, float ridge_eps, int max_iter, float tol, int lanczos_steps) {
  constexpr float kTopMin = 0.7f, kEnd = 0.97f;
  const int z = blockIdx.x, lane = threadIdx.x;
  const RootGroup& g = G.g[root_group_of(G, z)];
  const int p = g.p;
  const float part = G.st.partial[z * RCHUNKS + lane];
  float nrm2 = 0.f;
#pragma unroll
  for (int c = 0; c < RCHUNKS; ++c) nrm2 += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, part), c));
  const float sv = G.st.sv[z], zscale = (1.f + p) / (2.f * sqrtf(nrm2)), ridge = ridge_eps * sv;
  const float a0 = 1.f + 1.f / p, b0 = 1.f / p;
  float ca = a0, cb = b0;                      // of step `lane`
  int quartic = -1;                            // its row of kRootQuartics
  int k = 0;
  if (ridge_eps >= 1e-7f && p >= 2 && p <= 8 && max_iter >= kRootSteps && sv > 0.f && 0.5f * ridge * zscale > 1e-9f) {
    const int dim = G.st.lz_dim[z];
    const float low = lowest_ritz(G.st.alpha + z * kLanczosSteps, G.st.beta + z * kLanczosSteps, dim == 0 ? lanczos_steps : dim,
                                  ridge, 0.5f * ridge, sv + ridge);
    const float near = fmaxf(tol, 1e-6f);
    const int classical = max(classical_steps(low * zscale, p, a0, b0, near, 0),
                              classical_steps((sv + ridge) * zscale, p, a0, b0, near, 0));
    float l = fmaxf(0.5f * low, 0.5f * ridge) * zscale;
    const float cp = int_power(static_cast<float>(p) / (p + 1), p) / (p + 1);       // b = cp a^(p+1)
    // the classical steps: the spectrum is in [l, (1 + p) / 2], and in (0, 1] after the first
    const float first = 0.5f * (1 + p) * int_power(a0 - b0 * 0.5f * (1 + p), p);
    for (; k < kRootEarly; ++k) {
      l *= int_power(a0 - b0 * l, p);
      if (k == 0) l = fminf(l, first);
    }
    int cost = 4 * kRootEarly;                 // products of the schedule (a classical step takes four, one of the fourth degree six)
    if (g.quartic != 0) {
      // a row of the table per lane
      float row[6];
#pragma unroll
      for (int i = 0; i < 6; ++i) row[i] = kRootQuartics[min(lane, kRootQuarticRows - 1)][i];
      auto raised = [&](float m) {
        const float u = 2.f * m - 1.f, t2 = 2.f * u * u - 1.f, t3 = 2.f * u * t2 - u, t4 = 2.f * t2 * t2 - 1.f;
        return m * int_power(row[1] + row[2] * u + row[3] * t2 + row[4] * t3 + row[5] * t4, 4);
      };
      const float floor = lane == 0 ? kRootQuarticTop : raised(row[0]);
      int then = classical_steps(l, p, a0, b0, near, 0);
      while (k < kRootSteps - 1) {
        const unsigned long long fits = __ballot(lane < kRootQuarticRows && (lane == 0 || row[0] <= l));
        const int which = 63 - __clzll(fits);
        const float next = __shfl(fminf(raised(l), floor), which);
        const int after = classical_steps(next, p, a0, b0, near, 0);
        if (6 + 4 * max(after, 1) >= 4 * then) break;
        if (lane == k) quartic = which;
        ++k;
        cost += 6;
        l = next;
        then = after;
      }
      cost += 4 * max(then, 1);
    } else for (; k < kRootSteps - 1 && l < kEnd; ++k) {
      // the a in [1 + 1/p, 2.5] that maximises min(f(l), f(1)), f(m) = m (a - b m)^p: two rounds of 64 candidates
      float lo = a0, hi = 2.5f, a = a0, v = -1.f;
#pragma unroll
      for (int round = 0; round < 2; ++round) {
        const float c = lo + (hi - lo) * (lane / 63.f);
        const float ap = int_power(c, p), b = cp * ap * c;
        const float top = int_power(c - b, p), low_end = l * int_power(c - b * l, p);
        const float value = c > b && ap <= 12.f && (top >= kTopMin || c == a0) ? fminf(top, low_end) : -1.f;
        const float best = wave_max(value);
        const int who = __ffsll(__ballot(value == best)) - 1;
        a = __shfl(c, who);
        v = best;
        const float h = (hi - lo) / 63.f;
        lo = fmaxf(a0, a - h);
        hi = a + h;
      }
      if (!(v > l)) break;
      if (lane == k) {
        ca = a;
        cb = cp * int_power(a, p) * a;
      }
      l = v;
    }
    if (g.quartic != 0 ? cost >= 4 * classical : classical_steps(l, p, a0, b0, near, k) >= classical) {
      k = 0;
      ca = a0;
      cb = b0;
      quartic = -1;
    }
  }
  if (lane < kRootSteps) {
    float* __restrict__ coef = G.st.coef + (z * kRootSteps + lane) * kCoefs;
    if (quartic >= 0) {
      const float* __restrict__ c = kRootQuartics[quartic] + 1;
      coef[2] = 2.f * c[3];
      coef[3] = 4.f * c[4];
      coef[4] = c[0] - c[4] - 1.f;
      coef[5] = c[1] - c[3];
      coef[6] = c[2];
      ca = -1.f;                               // the matrix that the products of such a step start from is U = 2 M - I
      cb = -2.f;
    }
    // the steps behind the early ones take T - I where they may be of the fourth degree
    coef[0] = g.quartic != 0 && k > 0 && lane >= k ? ca - 1.f : ca;
    coef[1] = cb;
  }
  if (lane == 0) {
    G.st.accel[z] = k;
    G.st.zscale[z] = zscale;
  }
}

// grid (RCHUNKS, total), fp32 groups: M = z S, T = a I - b M and the X of the first step, z^(1/p) T (X_0 is a multiple of the
// identity and never stored); the padding columns are zero; partial max |M - I|
static __global__ __launch_bounds__(256) void root_start_kernel(RootGroups G) {
  __shared__ float red[4];
  const int z = blockIdx.y;
  const RootGroup& g = G.g[root_group_of(G, z)];
  if (g.np != 0) return;
  const int n = g.n, ld = g.ld;
  const float zs = G.st.zscale[z], r0 = powf(zs, 1.0f / g.p);
  const float a = G.st.coef[z * kCoefs * kRootSteps], b = G.st.coef[z * kCoefs * kRootSteps + 1];
  const int64_t mat = static_cast<int64_t>(n) * ld, buf = mat * g.batch;
  const float* __restrict__ S = g.S + (z - g.z0) * g.strideS;
  float* __restrict__ base = g.bufs + (z - g.z0) * mat;
  float e = 0.f;
  const int lane = threadIdx.x & 63;
  for (int i = 4 * blockIdx.x + (threadIdx.x >> 6); i < n; i += 4 * RCHUNKS) {
#pragma unroll 4
    for (int j = lane; j < ld; j += 64) {
      const bool inside = j < n, diag = i == j;
      const float m = inside ? zs * S[static_cast<int64_t>(i) * n + j] : 0.f;
      const float t = (diag ? a : 0.f) - b * m;
      const int64_t at = static_cast<int64_t>(i) * ld + j;
      base[buf + at] = r0 * t;
      base[2 * buf + at] = m;
      base[4 * buf + at] = t;
      if (!inside)                             // no product writes the padding columns
        for (int k = 0; k < g.buffers; ++k) base[k * buf + at] = 0.f;
      if (inside) e = fmaxf(e, fabsf(m - (diag ? 1.f : 0.f)));
    }
  }
  e = wave_max(e);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) G.st.partial[z * RCHUNKS + blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// grid (RCHUNKS, batch): the same on planes over the padded index range (zero outside n x n).  NP = 2 (fp16 planes): M and T
// scaled by kRootScaleM, X without its factor z^(1/p): scale_r T.
template <int NP>
static __global__ __launch_bounds__(256) void root_start_planes_kernel(RootState st, RootGroup g) {
  __shared__ float red[4];
  const int zl = blockIdx.y, z = g.z0 + zl;
  const float zs = st.zscale[z];
  const float r0 = NP == 2 ? g.scale_r : powf(zs, 1.0f / g.p);
  const float sm = NP == 2 ? kRootScaleM : 1.f;
  const float a = st.coef[z * kCoefs * kRootSteps], b = st.coef[z * kCoefs * kRootSteps + 1];
  const int n = g.n, n_pad = g.n_pad;
  const int64_t plane = static_cast<int64_t>(n_pad) * n_pad, set = NP * plane, buf = set * g.batch;
  const float* __restrict__ S = g.S + zl * g.strideS;
  unsigned short* __restrict__ base = reinterpret_cast<unsigned short*>(g.bufs) + zl * set;
  float e = 0.f;
  const int lane = threadIdx.x & 63;
  for (int i = 4 * blockIdx.x + (threadIdx.x >> 6); i < n_pad; i += 4 * RCHUNKS) {
    for (int j = 4 * lane; j < n_pad; j += 256) {
      floatx4 x = {0.f, 0.f, 0.f, 0.f};
      const float* src = S + static_cast<int64_t>(i) * n + j;
      if (i < n && j + 4 <= n) {
        x = *reinterpret_cast<const floatx4u*>(src);
      } else if (i < n) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
          if (j + k < n) x[k] = src[k];
      }
      u16x4 om[NP], ot[NP], ox[NP];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool inside = i < n && j + k < n, diag = i == j + k;
        const float m = zs * x[k], t = inside ? (diag ? a : 0.f) - b * m : 0.f;
        if (inside) e = fmaxf(e, fabsf(m - (diag ? 1.f : 0.f)));
        unsigned short o[3];
        plane_bits<NP>(m * sm, o);
#pragma unroll
        for (int q = 0; q < NP; ++q) om[q][k] = o[q];
        plane_bits<NP>(t * sm, o);
#pragma unroll
        for (int q = 0; q < NP; ++q) ot[q][k] = o[q];
        plane_bits<NP>(r0 * t, o);
#pragma unroll
        for (int q = 0; q < NP; ++q) ox[q][k] = o[q];
      }
      const int64_t dst = plane_index(i, j, n_pad);
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        *reinterpret_cast<u16x4*>(base + buf + q * plane + dst) = ox[q];
        *reinterpret_cast<u16x4*>(base + 2 * buf + q * plane + dst) = om[q];
        *reinterpret_cast<u16x4*>(base + 4 * buf + q * plane + dst) = ot[q];
      }
    }
  }
  e = wave_max(e);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) st.partial[z * RCHUNKS + blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// grid (total), one wave
static __global__ void root_begin_kernel(RootState st, float tol, int max_iter) {
  const int z = blockIdx.x;
  const float e = wave_max(st.partial[z * RCHUNKS + threadIdx.x]);
  if (threadIdx.x != 0) return;
  st.err[z] = e;
  st.active[z] = (e > tol && max_iter > 0) ? 1 : 0;
}

// (with `quartic`, the steps of the matrix's table in front of the classical ones; 0: every step is plain)
__device__ __forceinline__ int root_step_kind(int steps, int quartic) {
  return quartic == 0 || steps < kRootEarly ? kStepPlain : (steps < quartic ? kStepQuartic : kStepLate);
}

// A matrix's own state of the iteration.
struct RootProgress {
  float err;
  int count, active;
};
// Accepts or rejects the step whose products have run and decides whether to go on.  z: the entry with the state before the
// step and with the words that the step has folded into.  All lanes of a wave call it.
__device__ __forceinline__ RootProgress newton_decide(const RootState& st, int z, int accel, float tol, int max_iter) {
  RootProgress r{st.err[z], st.count[z], st.active[z]};
  const int overflow = st.ovf[z];
  uint32_t bits = __builtin_bit_cast(uint32_t, st.errword[(z * kErrSlots + (threadIdx.x & (kErrSlots - 1))) * kErrStride]);
#pragma unroll
  for (int o = kErrSlots / 2; o > 0; o >>= 1) bits = max(bits, static_cast<uint32_t>(__shfl_xor(static_cast<int>(bits), o)));
  const float e = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(bits));
  if (r.active == 0) return r;
  // diverging: keep the previous root (NaN compares false, like the reference).  The error of an accelerated step may grow, but
  // not beyond that of a spectrum in [0, 1].  A step whose products left the range of the fp16 planes (a statistic far
  // from positive definite) is dropped the same way.
  const float limit = r.count >= kRootEarly && r.count < accel ? 1.2f : r.err * 1.2f;
  if (overflow != 0 || e > limit) {
    r.active = 0;
    return r;
  }
  r.err = e;
  ++r.count;
  if (!(e > tol && r.count < max_iter)) r.active = 0;
  return r;
}

// grid (total), one wave: the decision about the step in half `half`, into the first half; all words are cleared.
static __global__ __launch_bounds__(64) void newton_decide_kernel(RootState st, int half, float tol, int max_iter) {
  const int z = blockIdx.x;
  const float last = st.settled[z];
  const int steps = st.count[half * st.total + z];
  RootProgress r = newton_decide(st, half * st.total + z, st.accel[z], tol, max_iter);
  if (threadIdx.x != 0) return;
  if (last > 0.f && r.count > steps) r.err = last;       // (that step had X' alone, which leaves no error behind)
  st.settled[z] = 0.f;
  st.err[z] = r.err;
  st.count[z] = r.count;
  st.active[z] = r.active;
  root_clear_words(st, z);
  root_clear_words(st, st.total + z);
}

// The last step in sight: M' = I - (5/8) E^2 - O(E^3), E = M - I, for p = 4, and |(E^2)_ij| is at most the largest squared length of a row
// of E.  Where that is tol or less the coming step ends the iteration by the very test of the reference, max |M' - I| <= tol (5/8 tol
// and the rounding of M', 2.4e-7), and its products T^2, T^2 M and M' are left out: three of 45, 11 ms of 98 statistics'
// 122, for one reading of M, 0.3 ms.
// grid (blocks of 32 columns, batch), behind a decision, groups on 192-wide tiles.  Bound by the memory: a wave reads 512 consecutive bytes.
static __global__ __launch_bounds__(256) void root_settled_kernel(RootState st, RootGroup g, float tol) {
  __shared__ float part[4][32];
  const int z = g.z0 + blockIdx.y, steps = st.count[z], accel = st.accel[z];
  const float e = st.err[z];
  if (st.active[z] == 0 || root_step_kind(steps, accel) != kStepLate || !(e * e <= tol)) return;
  const int64_t plane = static_cast<int64_t>(g.n_pad) * g.n_pad, set = 2 * plane;
  const unsigned short* __restrict__ M = reinterpret_cast<const unsigned short*>(g.bufs) + (2 + (steps & 1)) * set * g.batch +
                                         blockIdx.y * set + static_cast<int64_t>(blockIdx.x) * g.n_pad * 32;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = 4 * (lane & 7), j = 32 * blockIdx.x + col;
  floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int i = 8 * wave + (lane >> 3); i < g.n; i += 32) {
    const u16x4 hi = *reinterpret_cast<const u16x4*>(M + i * 32 + col), lo = *reinterpret_cast<const u16x4*>(M + plane + i * 32 + col);
    const floatx4 m = plane_values(hi, lo, 1.f / kRootScaleM);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float d = m[k] - (i == j + k ? 1.f : 0.f);
      sum[k] = __builtin_fmaf(d, d, sum[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    sum[k] += __shfl_xor(sum[k], 8);
    sum[k] += __shfl_xor(sum[k], 16);
    sum[k] += __shfl_xor(sum[k], 32);
    if (lane < 8) part[wave][col + k] = sum[k];
  }
  __syncthreads();
  if (tid >= 64) return;
  const int c = lane & 31;
  const float largest = wave_max((part[0][c] + part[1][c]) + (part[2][c] + part[3][c]));
  // (a NaN stays out; too long a row makes the word negative for good: as an unsigned number it is above all others)
  const bool fits = largest <= tol;
  if (lane == 0) atomicMax(reinterpret_cast<uint32_t*>(st.settled + z), __builtin_bit_cast(uint32_t, fits ? fmaxf(0.625f * largest, 1e-30f) : -1.f));
}

// grid (RCHUNKS, total): the caller's fp32 result
static __global__ __launch_bounds__(256) void root_out_kernel(RootGroups G) {
  const int z = blockIdx.y;
  const RootGroup& g = G.g[root_group_of(G, z)];
  const int zl = z - g.z0, n = g.n, count = G.st.count[z], lane = threadIdx.x & 63;
  float* __restrict__ out = g.out + zl * g.strideOut;
  const float r0 = powf(G.st.zscale[z], 1.0f / g.p);
  const int64_t mat = static_cast<int64_t>(n) * g.ld;
  const float* __restrict__ R = g.bufs + (count & 1) * mat * g.batch + zl * mat;
  const int64_t plane = static_cast<int64_t>(g.n_pad) * g.n_pad, set = g.np * plane;
  const unsigned short* __restrict__ P = reinterpret_cast<const unsigned short*>(g.bufs) + (count & 1) * set * g.batch + zl * set;
  // fp16 planes hold scale_r times the root without its factor z^(1/p); the sum of the bf16 planes is the root
  const float mul = r0 / g.scale_r;
  for (int i = 4 * blockIdx.x + (threadIdx.x >> 6); i < n; i += 4 * RCHUNKS) {
    for (int j = 4 * lane; j < n; j += 256) {
      floatx4 v;
      if (count == 0) {                           // no step was accepted
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = i == j + k ? r0 : 0.f;
      } else if (g.np == 0) {
        v = *reinterpret_cast<const floatx4*>(R + static_cast<int64_t>(i) * g.ld + j);
      } else {
        const int64_t src = plane_index(i, j, g.n_pad);
        u16x4 o[3];
#pragma unroll
        for (int q = 0; q < 3; ++q)
          if (q < g.np) o[q] = *reinterpret_cast<const u16x4*>(P + q * plane + src);
#pragma unroll
        for (int k = 0; k < 4; ++k)
          v[k] = g.np == 2 ? mul * (static_cast<float>(__builtin_bit_cast(_Float16, static_cast<unsigned short>(o[0][k]))) +
                                    static_cast<float>(__builtin_bit_cast(_Float16, static_cast<unsigned short>(o[1][k]))))
                           : (static_cast<float>(__builtin_bit_cast(__bf16, static_cast<unsigned short>(o[0][k]))) +
                              static_cast<float>(__builtin_bit_cast(__bf16, static_cast<unsigned short>(o[1][k])))) +
                                 static_cast<float>(__builtin_bit_cast(__bf16, static_cast<unsigned short>(o[2][k])));
      }
      float* dst = out + static_cast<int64_t>(i) * n + j;
      if (j + 4 <= n) {
        *reinterpret_cast<floatx4u*>(dst) = v;
      } else {
#pragma unroll
        for (int k = 0; k < 3; ++k)
          if (j + k < n) dst[k] = v[k];
      }
    }
  }
}

// grid (total)
static __global__ void root_stats_kernel(RootGroups G) {
  const int z = blockIdx.x;
  if (threadIdx.x != 0) return;
  const RootGroup& g = G.g[root_group_of(G, z)];
  float* __restrict__ stats = g.stats + 4 * (z - g.z0);
  stats[0] = G.st.sv[z];
  stats[1] = static_cast<float>(G.st.pi_iters[z]);
  stats[2] = static_cast<float>(G.st.count[z]);
  stats[3] = G.st.err[z];
}

// ---- products on small tiles ----------------------------------------------------------------------------------------------

enum RootKind { kFp32 = 0, kPlanes2 = 2, kPlanes3 = 3 };
// A product of a step, C = A B (b_late: of the steps behind the early ones of a matrix with steps of the fourth degree).
// next.index >= 0: it forms M', and writes the next step's polynomial, or the U that it starts from, and the error.
struct RootOp {
  PairedBuf a, b, c, next, b_late{-1, 0}, second{-1, 0}, u{-1, 0}, p{-1, 0};      // second, u, p: of the epilogue
  int epi = kEpiPlain;
  float shift_u = 0.f, shift_i = 0.f;
};
struct RootJob {
  float* bufs;                  // of its group
  int64_t buf_elems, mat_elems; // floats (planes: 16-bit elements) between buffers, between matrices
  RootOp op;
  int n, ld;                    // ld: padded size on planes
  int z0, tiles;                // first matrix; tiles of one matrix: on planes those on one side of the diagonal
  int kind;
  int quartic;                  // steps of the fourth degree are among its group's products
  float scale_r;
};
// (What leads a work group to its matrix lies side by side: the matrix's step count is then requested beside the job, whose
// address depends on it, and not a trip to memory after it.)
constexpr int kRootMaxJobs = 2 * kRootMaxGroups;
struct RootJobs {
  int first[kRootMaxJobs];      // first work group of each job, INT32_MAX behind the last
  int tiles[kRootMaxJobs], z0[kRootMaxJobs];
  RootJob j[kRootMaxJobs];
};

// One tile (ti, tj) of C = A B of fp32 matrices: every tile of the product (nothing is mirrored), k pairs (16 t + m, 16 t + 8 + m)
// in order on one accumulator, chunks of 128 k, the chunks added in order through the LDS.  THREADS = 1024 (512): 64 x 64, wave
// (q, w) sums chunk q of every four (two) of block w.  THREADS = 256 (launches without planes): 32 x 32, wave q sums chunk q of
// every four, so that few columns still spread over the device.  Operands go from memory to registers as the matrix instruction wants them.
// Bound by latency and, in the 64 x 64 form, by the fp32 matrix instruction (1.7 us per chunk and CU).
// EPI other than plain: U, P, the second result and the coefficients in `further`.
struct RootFurther {
  const float* U;
  const float* P;
  float* second;
  QuarticCoefs qc;
};
template <int THREADS, int EPI>
__device__ __forceinline__ float root_tile_fp32(const GemmParams& p, const RootFurther& further, int ti, int tj, AK_LDS floatx4* part) {
  constexpr int BLOCKS = THREADS == 256 ? 1 : 4, GROUPS = THREADS / 64 / BLOCKS, TILE = BLOCKS == 4 ? 64 : 32;
  constexpr int U = BLOCKS == 4 ? 2 : 4;                      // steps of 16 k loaded at once
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), q = wave / BLOCKS, w = wave % BLOCKS;
  const int i0 = TILE * ti + 32 * (w >> 1), j0 = TILE * tj + 32 * (w & 1), ld = static_cast<int>(p.lda);
  const bool col_in = j0 + l32 < p.M;
  const float* __restrict__ A = p.A + static_cast<int64_t>(i0 + l32 < p.M ? i0 + l32 : 0) * ld;
  const float* __restrict__ B = p.B + (col_in ? j0 + l32 : 0);
  const int chunks = (p.M + 127) / 128;
  floatx4 tot[4 / GROUPS];
#pragma unroll
  for (int k = 0; k < 4 / GROUPS; ++k) tot[k] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int first = 0; first < chunks; first += GROUPS) {
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    const int k1 = min(p.M, 128 * (first + q + 1));
    for (int k0 = 128 * (first + q); k0 < k1; k0 += 16 * U) {
      floatx4 a[U][2];
      float b[U][8];
      // (loads without conditions: each of those would be waited for by itself.  Rows and columns beyond the matrix read
      // others, whose sums are not stored; k beyond it are replaced by zeros.)
      const bool whole = k0 + 16 * U <= p.M;
#pragma unroll
      for (int t = 0; t < U; ++t) {
        const int k = k0 + 16 * t + 8 * g;
#pragma unroll
        for (int h = 0; h < 2; ++h) a[t][h] = *reinterpret_cast<const floatx4*>(A + (whole ? k + 4 * h : min(k + 4 * h, ld - 4)));
#pragma unroll
        for (int m = 0; m < 8; ++m) b[t][m] = B[static_cast<int64_t>(whole ? k + m : min(k + m, p.M - 1)) * ld];
      }
      if (!whole) {
#pragma unroll
        for (int t = 0; t < U; ++t)
#pragma unroll
          for (int m = 0; m < 8; ++m) {
            const bool in = k0 + 16 * t + 8 * g + m < p.M;
            a[t][m >> 2][m & 3] = in ? a[t][m >> 2][m & 3] : 0.f;
            b[t][m] = in ? b[t][m] : 0.f;
          }
      }
#pragma unroll
      for (int t = 0; t < U; ++t)
#pragma unroll
        for (int m = 0; m < 8; ++m) acc = mfma_f32(a[t][m >> 2][m & 3], b[t][m], acc);
    }
    add_chunks<BLOCKS, GROUPS>(acc, tot, first, chunks, q, w, GROUPS, part);
    if (first + GROUPS < chunks) __syncthreads();
  }
  float vmax = 0.f;
  if (col_in) {
#pragma unroll
    for (int r = 0; r < 16 / GROUPS; ++r) {
      const float v = tot[r >> 2][r & 3];
      const int gi = i0 + 8 * (q * (4 / GROUPS) + (r >> 2)) + 4 * g + (r & 3), gj = j0 + l32;
      if (gi >= p.M) continue;
      if constexpr (EPI != kEpiPlain) {
        const int64_t at = static_cast<int64_t>(gi) * ld + gj;
        const float u = further.U[at];
        p.C[at] = quartic_first<EPI>(further.qc, v, u, EPI == kEpiQuartic ? further.P[at] : 0.f, gi == gj);
        if constexpr (EPI == kEpiSquare) further.second[at] = quartic_second(further.qc, v, u, gi == gj);
        continue;
      }
      p.C[static_cast<int64_t>(gi) * ld + gj] = v;
      vmax = gemm_fold_absmax(vmax, v, gi == gj, 1);
      if (p.C2 != nullptr) p.C2[static_cast<int64_t>(gi) * ld + gj] = p.c2_scale * v + (gi == gj ? p.c2_diag : 0.f);
    }
  }
  return vmax;
}

// A product on planes (fp16 planes: the two roots carry scale_r, every other matrix kRootScaleM).
__host__ __device__ inline PlaneGemm root_plane_gemm(const RootState& st, int z0, int np, int n, int n_pad, int tile, float scale_r,
                                                     float* bufs, int64_t buf_elems, const RootOp& op, int quartic) {
  PlaneGemm pg;
  pg.bufs = reinterpret_cast<__bf16*>(bufs);
  pg.plane_elems = static_cast<int64_t>(n_pad) * n_pad;
  pg.set_elems = np * pg.plane_elems;
  pg.buf_elems = buf_elems;
  pg.A = op.a; pg.B = op.b; pg.C = op.c; pg.C2 = op.epi == kEpiPlain ? op.next : op.second;
  pg.B_late = op.b_late; pg.U = op.u; pg.P = op.p; pg.epi = op.epi;
  pg.u_scale = op.u.index == 0 ? scale_r : kRootScaleM;
  pg.shift_u = op.shift_u; pg.shift_i = op.shift_i;
  pg.count = st.count + z0;
  pg.accel = st.accel + z0;
  pg.early = quartic != 0 ? kRootEarly : 0;
  pg.coef = st.coef + static_cast<int64_t>(z0) * kCoefs * kRootSteps;
  pg.coef_stride = kCoefs * kRootSteps; pg.coef_last = kRootSteps - 1;
  pg.errword = op.next.index >= 0 ? st.errword + z0 * kErrSlots * kErrStride : nullptr;
  pg.active = st.active + z0;
  pg.settled = quartic != 0 && op.c.index != 0 ? st.settled + z0 : nullptr;
  pg.overflow = st.ovf + z0;
  pg.n = n; pg.n_pad = n_pad; pg.T = n_pad / tile;
  const float sa = op.a.index == 0 ? scale_r : kRootScaleM, sb = op.b.index == 0 ? scale_r : kRootScaleM;
  pg.in_unscale = 1.0f / (sa * sb);
  pg.c_scale = op.c.index == 0 ? scale_r : kRootScaleM;
  pg.c2_plane_scale = kRootScaleM;
  return pg;
}

__device__ __forceinline__ bool root_idle(const RootJob& job, int active, int steps, int kind) {
  return active == 0 || (steps == 0 && job.op.c.index == 0) ||       // (the first X is written by the start)
         ((job.op.epi == kEpiSquare || job.op.epi == kEpiQuartic) && kind != kStepQuartic);
}

// The product of matrix zl of a group in fp32; c2_*: of the step `steps` is followed by.
__device__ __forceinline__ GemmParams root_fp32_product(const RootState& st, const RootJob& job, int zl, int z, int steps, int kind) {
  const int parity = steps & 1;
  const RootOp& op = job.op;
  float* base = job.bufs + zl * job.mat_elems;
  GemmParams p;
  p.A = base + paired_buf(op.a, parity, kind) * job.buf_elems;
  p.B = base + paired_buf(op.b_late.index >= 0 && kind != kStepPlain ? op.b_late : op.b, parity, kind) * job.buf_elems;
  p.C = base + paired_buf(op.c, parity, kind) * job.buf_elems;
  p.lda = p.ldb = p.ldc = job.ld;
  p.M = p.N = job.n;
  p.K = job.ld;
  p.transB = 1;                 // (a symmetric operand is its own transpose)
  p.tile_mode = TILE_ALL;
  if (op.next.index >= 0) {
    const float* next = st.coef + (z * kRootSteps + min(steps + 1, kRootSteps - 1)) * kCoefs;
    p.C2 = base + paired_buf(op.next, parity, kind) * job.buf_elems;
    p.ldc2 = job.ld;
    p.c2_diag = next[0];
    p.c2_scale = -next[1];
    p.absmax_out = st.errword + (z * kErrSlots + blockIdx.x % kErrSlots) * kErrStride;
    p.absmax_identity = 1;
  }
  return p;
}

// Products of a group in fp32 with many wide matrices: 128 x 128 tiles of the three-piece split (gemm_x3.hpp).
static __global__ __launch_bounds__(256) void root_split_kernel(RootState st, RootJob job) {
  __shared__ __attribute__((aligned(16))) unsigned char x3_smem[2 * 2 * 3 * X3_PLANE];
  const int zl = static_cast<int>(blockIdx.x) / job.tiles, z = job.z0 + zl, local = static_cast<int>(blockIdx.x) - zl * job.tiles;
  const int steps = st.count[z], T = (job.n + X3_BT - 1) / X3_BT;
  if (root_idle(job, st.active[z], steps, kStepPlain)) return;
  GemmParams p = root_fp32_product(st, job, zl, z, steps, kStepPlain);
  p.K = job.n;
  p.transB = 0;
  gemm_x3_tile<3, true, 1, 0, false, true>(p, local / T, local % T, 0, (AK_LDS3 unsigned char*)x3_smem);
}

// A tile's largest |M' - I| and whether it fits, folded into entry z, word `slot`.
__device__ __forceinline__ void root_fold(const RootState& st, int z, int slot, float vmax, bool fits) {
  __shared__ uint32_t largest[16], lost[16];
  uint32_t bits = __builtin_bit_cast(uint32_t, fabsf(vmax));            // a NaN is larger than any number
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) bits = max(bits, static_cast<uint32_t>(__shfl_xor(static_cast<int>(bits), o)));
  const bool out = __ballot(!fits) != 0;
  if ((threadIdx.x & 63) == 0) {
    largest[threadIdx.x >> 6] = bits;
    lost[threadIdx.x >> 6] = out ? 1u : 0u;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  uint32_t any = 0;
  for (unsigned w = 0; w < blockDim.x / 64; ++w) {
    bits = max(bits, largest[w]);
    any |= lost[w];
  }
  atomicMax(reinterpret_cast<uint32_t*>(st.errword + (z * kErrSlots + slot) * kErrStride), bits);
  if (any != 0) atomicOr(st.ovf + z, 1);
}

// One step of the product sequences of all groups on small tiles: a work group per tile of any product.  THREADS = 256: no
// product on planes among them; 512: more tiles than CUs (two work groups a CU), 1024 else.
// Where all products of a call run here the steps need no launch for their decisions (5 us each): the first launch of a step
// (pending) takes the one about the step before, every work group for itself, from the half of the state that step used; one work
// group per matrix writes the new state to the other half, `half`, which the step's further launches read.  The words of
// the half that the next step will fold into are cleared by the last launch of a step: nothing else touches them then.
template <int THREADS>
static __global__ __launch_bounds__(THREADS, THREADS == 256 ? 1 : 4) void root_small_kernel(RootState st, RootJobs J, int half,
                                                                                            int pending, float tol, int max_iter) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char dtl_smem[];
  const int wg = static_cast<int>(xcd_contiguous_id(blockIdx.x, gridDim.x));      // a matrix's tiles share an L2
  int ji = 0, start = J.first[0], tiles = J.tiles[0], z0 = J.z0[0];
#pragma unroll
  for (int k = 1; k < kRootMaxJobs; ++k) {
    const bool here = wg >= J.first[k];
    ji = here ? k : ji;
    start = here ? J.first[k] : start;
    tiles = here ? J.tiles[k] : tiles;
    z0 = here ? J.z0[k] : z0;
  }
  const int zl = (wg - start) / tiles, z = z0 + zl, local = wg - start - zl * tiles;
  const int entry = half * st.total + z;
  const RootJob job = J.j[ji];
  const int accel = st.accel[z];
  int steps, active;
  if (pending != 0) {
    const RootProgress r = newton_decide(st, (1 - half) * st.total + z, accel, tol, max_iter);
    steps = r.count;
    active = r.active;
    if (local == 0 && job.op.c.index != 0 && threadIdx.x == 0) {
      st.err[entry] = r.err;
      st.count[entry] = r.count;
      st.active[entry] = r.active;
    }
  } else {
    steps = st.count[entry];
    active = st.active[entry];
  }
  steps = __builtin_amdgcn_readfirstlane(steps);
  const int kind = root_step_kind(steps, job.quartic != 0 ? __builtin_amdgcn_readfirstlane(accel) : 0);
  if (root_idle(job, __builtin_amdgcn_readfirstlane(active), steps, kind)) return;
  float vmax = 0.f;
  bool fits = true;
  if (THREADS == 256 || job.kind == kFp32) {
    const int T = (job.n + (THREADS == 256 ? 31 : 63)) / (THREADS == 256 ? 32 : 64);
    const GemmParams p = root_fp32_product(st, job, zl, z, steps, kind);
    RootFurther f = {};
    if (job.op.epi == kEpiPlain || (job.op.epi == kEpiShifted && kind == kStepPlain)) {
      vmax = root_tile_fp32<THREADS, kEpiPlain>(p, f, local / T, local % T, (AK_LDS floatx4*)dtl_smem);
    } else {
      float* base = job.bufs + zl * job.mat_elems;
      f.U = base + paired_buf(job.op.u, steps & 1, kind) * job.buf_elems;
      f.qc = quartic_coefs(st.coef + (z * kRootSteps + min(steps, kRootSteps - 1)) * kCoefs);
      if (job.op.epi == kEpiShifted) {
        f.qc = QuarticCoefs{0.f, 0.f, job.op.shift_i, job.op.shift_u, 0.f};
        root_tile_fp32<THREADS, kEpiShifted>(p, f, local / T, local % T, (AK_LDS floatx4*)dtl_smem);
      } else if (job.op.epi == kEpiSquare) {
        f.second = base + paired_buf(job.op.second, steps & 1, kind) * job.buf_elems;
        root_tile_fp32<THREADS, kEpiSquare>(p, f, local / T, local % T, (AK_LDS floatx4*)dtl_smem);
      } else {
        f.P = base + paired_buf(job.op.p, steps & 1, kind) * job.buf_elems;
        root_tile_fp32<THREADS, kEpiQuartic>(p, f, local / T, local % T, (AK_LDS floatx4*)dtl_smem);
      }
    }
  } else {
    int ti, tj;
    decode_lower_tile(local, ti, tj);
    const PlaneGemm pg = root_plane_gemm(st, job.z0, job.kind == kPlanes2 ? 2 : 3, job.n, job.ld, kPlaneSmallTile, job.scale_r,
                                         job.bufs, job.buf_elems, job.op, job.quartic);
    constexpr int GROUPS = THREADS == 512 ? 2 : 4;
    if (job.kind == kPlanes2) plane_tile_small<2, GROUPS>(pg, tj, ti, zl, steps, kind, (AK_LDS unsigned char*)dtl_smem, vmax, fits);
    else plane_tile_small<3, GROUPS>(pg, tj, ti, zl, steps, kind, (AK_LDS unsigned char*)dtl_smem, vmax, fits);
  }
  if (job.op.next.index >= 0) {
    if (local == 0 && threadIdx.x == 0) root_clear_words(st, (1 - half) * st.total + z);
    root_fold(st, entry, local % kErrSlots, vmax, fits);
  } else if (__ballot(!fits) != 0 && (threadIdx.x & 63) == 0) {
    atomicOr(st.ovf + entry, 1);
  }
}

// ---- host ----------------------------------------------------------------------------------------------------------

enum RootBuf { R0 = 0, M0 = 2, T0 = 4, B0 = 6 };
constexpr int kRootMaxSlots = 64;
constexpr PairedBuf kRin{R0, 1}, kRout{R0, 2}, kMin{M0, 1}, kMout{M0, 2}, kTin{T0, 1}, kTout{T0, 2}, kNone{-1, 0};
constexpr int kQuarticSlots = 2;        // products in front of the classical ones

// The products of one Newton step by slots: the products of a slot are independent of each other.  T^p by repeated
// squaring, with the multiplication order of the reference's MatPower for other powers.
// quartic (p = 4): two products in front that only steps of the fourth degree have, P = 2 U^2 - I with Y = y(U, P), then
// T = t(U, P) + P Y, which lies where the step's polynomial for the next one will; and behind the early steps M' is not
// (T^2)^2 M but (T^2 M) T^2: its rounding (at the top of the file), and T^4 of up to 29 would leave the range of the fp16 planes, whose
// scale of 2^12 ends at 16.
static int root_ops(int p, bool quartic, RootOp (*slots)[2], int* counts, int max_slots) {
  if (quartic) {
    const PairedBuf b0{B0, 0}, b1{B0 + 1, 0}, t{T0, 3};
    const RootOp ops[5] = {{kTin, kTin, b0, kNone, kNone, b1, kTin, kNone, kEpiSquare},
                           {b0, b1, kTout, kNone, kNone, kNone, kTin, b0, kEpiQuartic},
                           {t, t, b0, kNone, kNone, kNone, t, kNone, kEpiShifted, 2.f, 1.f},
                           {b0, b0, b1, kNone, kMin},
                           {b1, kMin, kMout, kTout, b0}};
    for (int k = 0; k < 5; ++k) {
      slots[k][0] = ops[k];
      counts[k] = 1;
    }
    slots[kQuarticSlots][1] = RootOp{kRin, t, kRout, kNone, kNone, kNone, kRin, kNone, kEpiShifted, 1.f, 0.f};
    counts[kQuarticSlots] = 2;
    return 5;
  }
  int n = 0;
  auto put = [&](PairedBuf a, PairedBuf b, PairedBuf c, PairedBuf c2) {
    if (n < max_slots) { slots[n][0] = RootOp{a, b, c, c2}; counts[n] = 1; }
    ++n;
  };
  auto same = [](PairedBuf x, PairedBuf y) { return x.index == y.index && x.sel == y.sel; };
  PairedBuf base = kTin, power = kNone;
  auto free_buf = [&] {
    for (int i = 0; i < 4; ++i) {
      const PairedBuf b{static_cast<int16_t>(B0 + i), 0};
      if (!same(b, base) && !same(b, power)) return b;
    }
    return PairedBuf{B0 + 3, 0};
  };
  for (int q = p; q > 0; q /= 2) {
    if (q & 1) {
      if (power.index < 0) {
        power = base;
      } else {
        const PairedBuf out = free_buf();
        put(base, power, out, kNone);
        power = out;
      }
    }
    if (q / 2 > 0) {
      const PairedBuf out = free_buf();
      put(base, base, out, kNone);
      base = out;
    }
  }
  put(power, kMin, kMout, kTout);                                  // M' = T^p M, its error, the next T
  if (n > max_slots) return -1;
  slots[0][1] = RootOp{kRin, kTin, kRout, kNone};                  // X' = X T, beside the first of them
  counts[0] = 2;
  return n;
}

// Buffers that the products of power p need: the fixed ones and the product buffers that root_ops() names.  0: p has too many steps.
static int root_buffers(int p) {
  RootOp slots[kRootMaxSlots][2];
  int counts[kRootMaxSlots];
  const int n = root_ops(p, false, slots, counts, kRootMaxSlots);       // (steps of the fourth degree take no buffer more)
  int most = kRootFixedBuffers;
  for (int k = 0; k < n; ++k)
    for (int o = 0; o < counts[k]; ++o)
      if (slots[k][o].c.sel == 0) most = std::max(most, slots[k][o].c.index + 1);
  return n < 0 ? 0 : most;
}

static size_t root_state_floats(int total) {
  return (static_cast<size_t>(total) * (4 + RCHUNKS + 2 * kLanczosSteps + kCoefs * kRootSteps + 2 * kErrSlots * kErrStride + 10) + 63) / 64 * 64;
}
// matrix buffers and Lanczos vectors of a group
static size_t root_group_matrix_floats(int64_t n, int64_t batch, int np, int buffers) {
  return (static_cast<size_t>(batch) * buffers * root_buffer_floats(n, batch, np) + 63) / 64 * 64;
}
static size_t root_group_floats(int64_t n, int64_t batch, int np, int buffers) {
  return root_group_matrix_floats(n, batch, np, buffers) + (static_cast<size_t>(5) * batch * n + 63) / 64 * 64;
}
static bool root_args_ok(const int64_t* n, const int* batch, int groups) {
  if (n == nullptr || batch == nullptr || groups <= 0 || groups > kRootMaxGroups) return false;
  int64_t total = 0;
  for (int i = 0; i < groups; ++i) {
    if (n[i] <= 0 || n[i] > (1 << 20) || batch[i] <= 0) return false;
    total += batch[i];
  }
  return total <= 65535;
}
// phases: 1 = power iteration, ridge and start of the Newton iteration; 2 = `iters` Newton iterations; 4 = results and
// statistics
static int root_run(int phases, int iters, RootGroups& G, float ridge_eps, int max_power_iter, float power_tol, int max_iter,
                    float tol, hipStream_t s) {
  const int total = G.total;
  const dim3 gz(total), gc(RCHUNKS, total), b256(256), b64(64);
  if (phases & 1) {
    const int steps = std::min(kLanczosSteps, std::max(1, max_power_iter));
    LanczosGroups L;
    int blocks = 0, widest = 0, narrowest = INT32_MAX;
    int64_t bytes = 0;
    for (int i = 0; i < kRootMaxGroups; ++i) {
      L.first[i] = i < G.count ? blocks : INT32_MAX;
      if (i >= G.count) continue;
      const RootGroup& g = G.g[i];
      L.g[i] = LanczosGroup{g.S, g.v0, g.vec, g.bufs, g.strideS, g.n, g.batch, g.z0, 0};
      blocks += g.batch * ((g.n + kLanczosRows - 1) / kLanczosRows);
      widest = std::max(widest, g.n);
      narrowest = std::min(narrowest, g.n);
      bytes += static_cast<int64_t>(4) * g.batch * g.n * g.n;
    }
    const bool wide = widest > kLanczosLdsDim, held = widest <= 1024 && blocks <= 512;       // (two work groups a CU)
    const size_t lds = static_cast<size_t>(widest) * sizeof(float);
    static bool attr_set = false;     // idempotent; a race sets it twice at worst
    if (!wide && lds > 60 * 1024 && !attr_set) {
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(root_lanczos_kernel<false, false>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              kLanczosLdsDim * static_cast<int>(sizeof(float))) != hipSuccess)
        return AK_ERR_LAUNCH;
      attr_set = true;
    }
    const bool half = lanczos_halves(widest, narrowest, bytes);
    if (half) {
      blocks = 0;
      for (int i = 0; i < G.count; ++i) {
        const int nb = (G.g[i].n + kLanczosTile - 1) / kLanczosTile;
        L.first[i] = blocks;
        blocks += G.g[i].batch * (nb * (nb + 1) / 2);
      }
      for (int j = 0; j <= steps; ++j) {
        hipLaunchKernelGGL(root_lanczos_vector_kernel, gz, dim3(1024), 0, s, G.st, L, j, steps);
        if (j < steps) hipLaunchKernelGGL(root_lanczos_tiles_kernel, dim3(blocks), b256, 0, s, G.st, L, j);
      }
    }
    for (int j = 0; j < steps && !half; ++j) {
      if (wide) hipLaunchKernelGGL((root_lanczos_kernel<true, false>), dim3(blocks), b256, 0, s, G.st, L, j);
      else if (held) hipLaunchKernelGGL((root_lanczos_kernel<false, true>), dim3(blocks), b256, lds, s, G.st, L, j);
      else hipLaunchKernelGGL((root_lanczos_kernel<false, false>), dim3(blocks), b256, lds, s, G.st, L, j);
    }
    hipLaunchKernelGGL(root_power_kernel, gz, b64, 0, s, G, steps, power_tol, max_power_iter);
    hipLaunchKernelGGL(root_ridge_kernel, gc, b256, 0, s, G, ridge_eps);
    hipLaunchKernelGGL(root_schedule_kernel, gz, b64, 0, s, G, ridge_eps, max_iter, tol, steps);
    bool fp32 = false;
    for (int i = 0; i < G.count; ++i) {
      const RootGroup& g = G.g[i];
      const dim3 gp(RCHUNKS, g.batch);
      if (g.np == 2) hipLaunchKernelGGL(root_start_planes_kernel<2>, gp, b256, 0, s, G.st, g);
      else if (g.np == 3) hipLaunchKernelGGL(root_start_planes_kernel<3>, gp, b256, 0, s, G.st, g);
      else fp32 = true;
    }
    if (fp32) hipLaunchKernelGGL(root_start_kernel, gc, b256, 0, s, G);
    hipLaunchKernelGGL(root_begin_kernel, gz, b64, 0, s, G.st, tol, max_iter);
  }
  if (phases & 2) {
    RootOp slots[kRootMaxGroups][kRootMaxSlots][2];
    int counts[kRootMaxGroups][kRootMaxSlots], nslots[kRootMaxGroups], most = 0;
    for (int i = 0; i < G.count; ++i) {
      nslots[i] = root_ops(G.g[i].p, G.g[i].quartic != 0, slots[i], counts[i], kRootMaxSlots);
      if (nslots[i] < 0) return AK_ERR_ARG;
      most = std::max(most, nslots[i]);
    }
    bool planes = false, small = true;          // products on planes among the small tiles; nothing but small tiles
    for (int i = 0; i < G.count; ++i) {
      const RootGroup& g = G.g[i];
      const bool on_small = g.np != 0 ? g.tile == kPlaneSmallTile : !root_split(g.n, g.batch);
      planes = planes || (g.np != 0 && on_small);
      // (with a single slot the first launch of a step is also its last)
      small = small && on_small && nslots[i] > 1;
    }
    const int edge = planes ? 64 : 32;                                               // of an fp32 tile
    // LDS by kind, with four and with two groups of waves
    constexpr int kLds[2][4] = {{65536, 0, kSmallTileLds<2, 4>, kSmallTileLds<3, 4>}, {32768, 0, kSmallTileLds<2, 2>, kSmallTileLds<3, 2>}};
    static bool attr_set = false;     // idempotent; a race sets it twice at worst
    if (!attr_set) {
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(root_small_kernel<1024>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              kLds[0][3]) != hipSuccess ||
          hipFuncSetAttribute(reinterpret_cast<const void*>(root_small_kernel<512>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              kLds[1][3]) != hipSuccess)
        return AK_ERR_LAUNCH;
      attr_set = true;
    }
    for (int it = 0; it < iters; ++it) {
      // (where the call's own first steps are known to be early, no products of the fourth degree are launched)
      const int skip = (phases & 1) != 0 && it < kRootEarly ? kQuarticSlots : 0;
      for (int slot = 0; slot < most; ++slot) {
        RootJobs J;
        int jobs = 0, blocks = 0, widest = 0;
        for (int i = 0; i < G.count; ++i) {
          const RootGroup& g = G.g[i];
          const int k = slot + (g.quartic != 0 ? skip : 0);
          if (k >= nslots[i]) continue;
          const int64_t mat = g.np == 0 ? static_cast<int64_t>(g.n) * g.ld : static_cast<int64_t>(g.np) * g.n_pad * g.n_pad;
          for (int o = 0; o < counts[i][k]; ++o) {
            RootOp op = slots[i][k][o];
            if (skip != 0) op.epi = kEpiPlain;
            if (g.np != 0 && g.tile == kPlaneTile) {
              const int rc = launch_plane_gemm(root_plane_gemm(G.st, g.z0, g.np, g.n, g.n_pad, g.tile, g.scale_r, g.bufs,
                                                               mat * g.batch, op, g.quartic), g.np, g.batch, s);
              if (rc != AK_OK) return rc;
              continue;
            }
            RootJob job;
            job.bufs = g.bufs; job.buf_elems = mat * g.batch; job.mat_elems = mat;
            job.op = op;
            job.quartic = g.quartic;
            job.n = g.n; job.ld = g.np == 0 ? g.ld : g.n_pad;
            job.z0 = g.z0;
            job.scale_r = g.scale_r;
            auto put = [&](int kind, int tiles) {
              job.kind = kind; job.tiles = tiles;
              J.first[jobs] = blocks; J.tiles[jobs] = tiles; J.z0[jobs] = g.z0;
              J.j[jobs++] = job;
              blocks += tiles * g.batch;
              widest = std::max(widest, kind);
            };
            if (g.np != 0) {
              const int t = g.n_pad / kPlaneSmallTile;
              put(g.np, t * (t + 1) / 2);
            } else if (root_split(g.n, g.batch)) {
              const int t = (g.n + 127) / 128;
              job.kind = kFp32; job.tiles = t * t;
              hipLaunchKernelGGL(root_split_kernel, dim3(job.tiles * g.batch), b256, 0, s, G.st, job);
            } else {
              const int t = (g.n + edge - 1) / edge;
              put(kFp32, t * t);
            }
          }
        }
        if (jobs == 0) continue;
        for (int i = jobs; i < kRootMaxJobs; ++i) {
          J.first[i] = INT32_MAX;
          J.tiles[i] = 1;
          J.z0[i] = 0;
        }
        const int half = small ? it & 1 : 0, pending = small && it > 0 && slot == 0 ? 1 : 0;
        if (!planes)
          hipLaunchKernelGGL(root_small_kernel<256>, dim3(blocks), b256, 16384, s, G.st, J, half, pending, tol, max_iter);
        else if (blocks > 256)
          hipLaunchKernelGGL(root_small_kernel<512>, dim3(blocks), dim3(512), kLds[1][widest], s, G.st, J, half, pending, tol, max_iter);
        else
          hipLaunchKernelGGL(root_small_kernel<1024>, dim3(blocks), dim3(1024), kLds[0][widest], s, G.st, J, half, pending, tol, max_iter);
      }
      if (small) continue;
      hipLaunchKernelGGL(newton_decide_kernel, gz, b64, 0, s, G.st, 0, tol, max_iter);
      if ((phases & 1) != 0 && it < kRootEarly) continue;
      for (int i = 0; i < G.count; ++i) {
        const RootGroup& g = G.g[i];
        if (g.quartic != 0 && g.np == 2 && g.tile == kPlaneTile)
          hipLaunchKernelGGL(root_settled_kernel, dim3(g.n_pad / 32, g.batch), b256, 0, s, G.st, g, tol);
      }
    }
    if (small && iters > 0) hipLaunchKernelGGL(newton_decide_kernel, gz, b64, 0, s, G.st, (iters - 1) & 1, tol, max_iter);
  }
  if (phases & 4) {
    hipLaunchKernelGGL(root_out_kernel, gc, b256, 0, s, G);
    hipLaunchKernelGGL(root_stats_kernel, gz, b64, 0, s, G);
  }
  return check_launch();
}

}  // namespace ak

// Workspace: the state of all matrices (the `active` words first), then the matrices of each group.
extern "C" size_t ak_inv_root_group_ws_bytes(const int64_t* n, const int* batch, const int* p, float ridge_eps, int groups) {
  if (!ak::root_args_ok(n, batch, groups) || p == nullptr) return 0;
  size_t floats = 0;
  int total = 0;
  for (int i = 0; i < groups; ++i) {
    const int buffers = p[i] >= 1 ? ak::root_buffers(p[i]) : 0;
    if (buffers == 0) return 0;
    floats += ak::root_group_floats(n[i], batch[i], ak::root_planes(n[i], p[i], ridge_eps), buffers);
    total += batch[i];
  }
  return (ak::root_state_floats(total) + floats) * sizeof(float);
}

extern "C" size_t ak_inv_root_group_active_offset(const int64_t*, const int*, int) { return 0; }

extern "C" int ak_inv_root_group(int phases, int iters, int groups, float* const* S, const int64_t* n,
                                 const int* batch, const int64_t* strideS, const int* p, float ridge_eps,
                                 const float* const* v0, int max_power_iter, float power_tol, int max_iter, float tol,
                                 float* const* out, const int64_t* strideOut, float* const* stats, void* ws,
                                 size_t ws_bytes, ak_stream_t stream) {
  using namespace ak;
  if (phases < 1 || phases > 7 || iters < 0 || S == nullptr || strideS == nullptr ||
      p == nullptr || v0 == nullptr || out == nullptr || strideOut == nullptr || stats == nullptr || !root_args_ok(n, batch, groups))
    return AK_ERR_ARG;
  const size_t need = ak_inv_root_group_ws_bytes(n, batch, p, ridge_eps, groups);
  if (need == 0) return AK_ERR_ARG;
  if (ws == nullptr || ws_bytes < need) return AK_ERR_WORKSPACE;
  RootGroups G;
  G.count = groups;
  G.total = 0;
  int total = 0;
  for (int i = 0; i < groups; ++i) total += batch[i];
  float* w = static_cast<float*>(ws) + root_state_floats(total);
  for (int i = 0; i < groups; ++i) {
    if (S[i] == nullptr || v0[i] == nullptr || out[i] == nullptr || stats[i] == nullptr || n[i] < 2 || p[i] < 1 ||
        strideS[i] < n[i] * n[i] || strideOut[i] < n[i] * n[i])
      return AK_ERR_ARG;
    RootGroup& g = G.g[i];
    g.S = S[i]; g.out = out[i]; g.v0 = v0[i]; g.stats = stats[i];
    g.strideS = strideS[i]; g.strideOut = strideOut[i];
    g.n = static_cast<int>(n[i]); g.ld = static_cast<int>(root_ld(n[i])); g.batch = batch[i]; g.p = p[i];
    g.z0 = G.total;
    g.tile = root_plane_dim(n[i]) ? root_plane_tile(n[i], batch[i]) : kPlaneSmallTile;
    g.n_pad = static_cast<int>(root_pad(n[i], g.tile));
    // two fp16 planes where the ridge bounds the root, else three bf16 planes; every part of a computation in parts gets
    // the same arguments, hence the same answer
    g.scale_r = root_fp16_scale(n[i], p[i], ridge_eps);
    g.np = root_planes(n[i], p[i], ridge_eps);
    g.quartic = p[i] == 4 && (g.np == 2 || (g.np == 0 && !root_split(n[i], batch[i]))) ? 1 : 0;
    g.buffers = root_buffers(p[i]);
    g.bufs = w;
    g.vec = w + root_group_matrix_floats(n[i], batch[i], g.np, g.buffers);
    w += root_group_floats(n[i], batch[i], g.np, g.buffers);
    G.total += batch[i];
  }
  w = static_cast<float*>(ws);
  RootState& st = G.st;
  auto ints = [&](int k) { int* r = reinterpret_cast<int*>(w); w += k; return r; };
  auto floats = [&](int64_t k) { float* r = w; w += k; return r; };
  st.total = total;
  st.active = ints(2 * total);
  st.count = ints(2 * total);
  st.accel = ints(total);
  st.ovf = ints(2 * total);
  st.lz_dim = ints(total);
  st.pi_iters = ints(total);
  st.sv = floats(total);
  st.err = floats(2 * total);
  st.settled = floats(total);
  st.zscale = floats(total);
  st.errword = floats(static_cast<int64_t>(2 * total) * kErrSlots * kErrStride);
  st.partial = floats(static_cast<int64_t>(total) * RCHUNKS);
  st.alpha = floats(static_cast<int64_t>(total) * kLanczosSteps);
  st.beta = floats(static_cast<int64_t>(total) * kLanczosSteps);
  st.coef = floats(static_cast<int64_t>(total) * kCoefs * kRootSteps);
  return root_run(phases, iters, G, ridge_eps, max_power_iter, power_tol, max_iter, tol,
                  static_cast<hipStream_t>(stream));
}

extern "C" int ak_inv_root_plane_format(int64_t n, int p, float ridge_eps) {
  if (n <= 0 || !ak::root_plane_dim(n)) return 0;
  return ak::root_fp16_scale(n, p, ridge_eps) > 0.f ? 2 : 3;
}

extern "C" int ak_inv_root_lanczos_halves(const int64_t* n, const int* batch, int groups) {
  if (!ak::root_args_ok(n, batch, groups)) return 0;
  int64_t bytes = 0;
  for (int i = 0; i < groups; ++i) bytes += 4 * batch[i] * n[i] * n[i];
  return ak::lanczos_halves(*std::max_element(n, n + groups), *std::min_element(n, n + groups), bytes) ? 1 : 0;
}

// (for any power and ridge: three planes, four product buffers)
extern "C" size_t ak_inv_root_ws_bytes(int64_t n, int batch) {
  if (!ak::root_args_ok(&n, &batch, 1)) return 0;
  const int np = ak::root_plane_dim(n) ? 3 : 0;
  return (ak::root_state_floats(batch) + ak::root_group_floats(n, batch, np, ak::kRootFixedBuffers + 4)) * sizeof(float);
}

extern "C" int ak_inv_root_newton(float* S, int64_t n, int batch, int64_t strideS, int p, float ridge_eps,
                                  const float* v0, int max_power_iter, float power_tol, int max_iter, float tol,
                                  float* out, int64_t strideOut, float* stats, void* ws, size_t ws_bytes,
                                  ak_stream_t stream) {
  return ak_inv_root_group(7, max_iter, 1, &S, &n, &batch, &strideS, &p, ridge_eps, &v0, max_power_iter, power_tol,
                           max_iter, tol, &out, &strideOut, &stats, ws, ws_bytes, stream);
}

extern "C" size_t ak_inv_root_active_offset(int64_t, int) { return 0; }

extern "C" int ak_inv_root_newton_part(int phases, int iters, float* S, int64_t n, int batch, int64_t strideS, int p,
                                       float ridge_eps, const float* v0, int max_power_iter, float power_tol,
                                       int max_iter, float tol, float* out, int64_t strideOut, float* stats, void* ws,
                                       size_t ws_bytes, ak_stream_t stream) {
  return ak_inv_root_group(phases, iters, 1, &S, &n, &batch, &strideS, &p, ridge_eps, &v0,
                           max_power_iter, power_tol, max_iter, tol, &out, &strideOut, &stats, ws, ws_bytes, stream);
}
