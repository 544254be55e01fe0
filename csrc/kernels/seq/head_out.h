// The outputs of a delta rule's rows: each head over its root mean square, times a weight, a gate's sigmoid and a scale.
#pragma once
#include "row_vec.h"

// 2^shift lanes a head, four columns each, all of their loads before the first sum.  (A wave a head with a column a load is bound by
// the loads it has in flight: 8,536 rows x 16 heads of 128 to bf16 62 -> 36 us, 37 at the rate of a copy; 6,700 x 16 of 64 35 -> 16)
template <typename TO>
__global__ __launch_bounds__(256) void head_out_kernel(const float* __restrict__ raw, const float* __restrict__ gate, int ldg,
                                                       const float* __restrict__ w, int w_hs, TO* __restrict__ out, int ldo, int H, int n,
                                                       float eps, float scale, int items, int shift) {
  const int lanes = 1 << shift, c = 4 * (threadIdx.x & (lanes - 1));
  const int item = (int)((blockIdx.x * 256 + threadIdx.x) >> shift);
  if (item >= items || c >= n) return;                       // (n = 4 lanes: whole heads)
  const int t = item / H, h = item % H;
  const RowVec<4> o = row_load<4>(raw + (size_t)item * n + c), g = row_load<4>(gate + (size_t)t * ldg + (size_t)h * n + c),
                  wc = row_load<4>(w + (size_t)h * w_hs + c);
  float ss = 0.f;
#pragma unroll
  for (int x = 0; x < 4; ++x) ss += o.v[x] * o.v[x];
  for (int d = 1; d < lanes; d <<= 1) ss += __shfl_xor(ss, d, 64);
  const float rs = 1.f / sqrtf(ss / (float)n + eps);
  RowVec<4> y;
#pragma unroll
  for (int x = 0; x < 4; ++x) y.v[x] = o.v[x] * rs * wc.v[x] * sigmoid_f(g.v[x]) * scale;
  row_store<4>(out + (size_t)t * ldo + (size_t)h * n + c, y);
}

// false: not such heads (32, 64, 128 or 256 columns) or not so aligned
template <typename TO>
inline bool head_out(const float* raw, const float* gate, int ldg, const float* w, int w_hs, TO* out, int ldo, int H, int n, float eps, float scale,
                     int items, hipStream_t s) {
  const int shift = n == 32 ? 3 : n == 64 ? 4 : n == 128 ? 5 : n == 256 ? 6 : -1;
  if (shift < 0 || (uintptr_t)raw % 16 || (uintptr_t)gate % 16 || ldg % 4 || (uintptr_t)w % 16 || (uintptr_t)out % (4 * sizeof(TO)) || ldo % 4)
    return false;
  const int per = 256 >> shift;
  hipLaunchKernelGGL((head_out_kernel<TO>), dim3((items + per - 1) / per), dim3(256), 0, s, raw, gate, ldg, w, w_hs, out, ldo, H, n, eps, scale, items, shift);
  return true;
}
