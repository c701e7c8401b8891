// One draw per row of a categorical distribution given by logits: the largest of p_i / q_i, q_i exponential random numbers.
// Two classes are compared by (logits_i - logits_j) - (log q_i - log q_j): the normalisation of p drops out, and so does an
// offset that all logits of a row share, before anything is rounded to its size (logits_i - log q_i at an offset of 1e6 has a
// spacing of 0.06: another class than softmax's in 1 % of the rows).
// Bound by the device memory: logits and random numbers are read once (8192 x 4096: 268 MB in 43 us, 6.2 TB/s) where softmax,
// normalisation, their checks, the quotient and the argmax made a dozen passes and launches.
#include "common.hpp"

namespace ak {

struct Best {
  float x, l;      // logit and log q of the best class so far
  int i;
};

// (the difference of two logits of -inf is NaN: the best so far stays)
__device__ __forceinline__ void best_of(Best& a, float x, float l, int i) {
  const float d = (x - a.x) - (l - a.l);
  if (d > 0.f || (d == 0.f && i < a.i)) a = Best{x, l, i};
}

// One wave per row (few classes) or one work group of four waves per row.
template <int WAVES>
static __global__ __launch_bounds__(256) void sample_categorical_kernel(const float* __restrict__ logits,
                                                                        const float* __restrict__ q, int64_t rows,
                                                                        int classes, int64_t* __restrict__ targets,
                                                                        int* __restrict__ invalid) {
  __shared__ Best part[4];
  __shared__ int part_bad[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row = WAVES == 1 ? static_cast<int64_t>(blockIdx.x) * 4 + wave : blockIdx.x;
  if (row >= rows) return;
  const float* __restrict__ x = logits + row * classes;
  const float* __restrict__ e = q + row * classes;
  const int t = WAVES == 1 ? lane : threadIdx.x;
  constexpr int N = 64 * WAVES;
  Best b{-INFINITY, 0.f, 0x7fffffff};
  int bad = 0;
  auto take = [&](float xc, float ec, int c) {
    bad |= xc < INFINITY ? 0 : 1;             // +inf and NaN: softmax of such a row is NaN
    best_of(b, xc, logf(ec), c);
  };
  const bool vec = classes % 4 == 0 && ((reinterpret_cast<uintptr_t>(logits) | reinterpret_cast<uintptr_t>(q)) & 15) == 0;
  if (vec) {
#pragma unroll 4
    for (int c = 4 * t; c < classes; c += 4 * N) {
      const floatx4 xv = *reinterpret_cast<const floatx4*>(x + c), ev = *reinterpret_cast<const floatx4*>(e + c);
#pragma unroll
      for (int u = 0; u < 4; ++u) take(xv[u], ev[u], c + u);
    }
  } else {
#pragma unroll 4
    for (int c = t; c < classes; c += N) take(x[c], e[c], c);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) best_of(b, __shfl_xor(b.x, o), __shfl_xor(b.l, o), __shfl_xor(b.i, o));
  if constexpr (WAVES > 1) {
    if (lane == 0) part[wave] = b;
    const int any_bad = __any(bad);
    if (lane == 0) part_bad[wave] = any_bad;
    __syncthreads();
    b = part[0];
    bad = part_bad[0] | part_bad[1] | part_bad[2] | part_bad[3];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) best_of(b, part[w].x, part[w].l, part[w].i);
  }
  if constexpr (WAVES == 1) bad = __any(bad);
  if (t == 0) {
    const bool none = b.i >= classes;         // every logit -inf (or NaN)
    targets[row] = none ? 0 : b.i;
    if (invalid != nullptr && (bad != 0 || none)) *invalid = 1;       // (all writers write the same)
  }
}

}  // namespace ak

extern "C" int ak_sample_categorical(const float* logits, const float* q, int64_t rows, int64_t classes, int64_t* targets,
                                     int* invalid, ak_stream_t stream) {
  if (logits == nullptr || q == nullptr || targets == nullptr || rows <= 0 || classes <= 0) return AK_ERR_ARG;
  if (classes > (1 << 30) || rows > 0x7fffffff) return AK_ERR_TOO_LARGE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // a wave covers 256 classes per step of four: up to 1024 classes one wave per row leaves no lane idle for long
  if (classes <= 1024)
    hipLaunchKernelGGL(ak::sample_categorical_kernel<1>, dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(256), 0, s, logits,
                       q, rows, static_cast<int>(classes), targets, invalid);
  else
    hipLaunchKernelGGL(ak::sample_categorical_kernel<4>, dim3(static_cast<unsigned>(rows)), dim3(256), 0, s, logits, q, rows,
                       static_cast<int>(classes), targets, invalid);
  return ak::check_launch();
}
