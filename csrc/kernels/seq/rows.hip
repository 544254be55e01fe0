// Row-wise kernels of the stateful models: group RMS norm (also as the residual update), embedding
// gather into the fp32 residual stream, activations between GEMMs, logit cap, K/V store with the key
// norm, and the routing of a mixture of experts.  All statistics and sums are fp32.
#include "seq_common.h"
#include "fls_seq.h"
#include "row_vec.h"

// ------------------------------------------------------------------------- group RMS norm
// one block per (row, group): sum of squares of D / groups columns, then the scaled row part
template <typename TO, int ADD>
__global__ __launch_bounds__(256) void group_rmsnorm_kernel(const float* __restrict__ x, int ldx, const int* __restrict__ idx,
                                                            const float* __restrict__ w, TO* __restrict__ y, int ldy,
                                                            int D, int groups, float eps, float woff, int w_one) {
  __shared__ float red[4];
  const int r = blockIdx.x, g = blockIdx.y;
  const int n = D / groups;
  const float* xr = x + (size_t)(idx != nullptr ? idx[r] : r) * ldx + (size_t)g * n;
  float ss = 0.f;
  for (int c = threadIdx.x; c < n; c += 256) { const float v = xr[c]; ss += v * v; }
  ss = block_sum_256(ss, red);
  const float rs = 1.f / sqrtf(ss / (float)n + eps);
  const float* wg = w + (size_t)g * n;
  TO* yr = y + (size_t)r * ldy + (size_t)g * n;
  for (int c = threadIdx.x; c < n; c += 256) {
    const float v = xr[c] * rs * ((w_one ? w[0] : wg[c]) + woff);
    if constexpr (ADD) yr[c] += v; else stf(yr, c, v);
  }
}

// The same with rows held in registers, four columns a thread and step: inputs and weights are read once, together, before the
// reduction.  MODE 0: y = norm(x); 1: y += norm(x); 2: y += norm(x), then h = norm(y; w2) of the new row: a sublayer's
// post-norm, the residual update and the next sublayer's norm in one pass.  Bound by its bytes from some hundred rows on
// and by a launch and two memory latencies below.  16384 rows of 4096 in two groups, a column a thread before: norm 146 -> 82 us,
// residual update 199 -> 140, update and next norm in turn 345, here 182.  SUM: x is a mixture's rows, sorted by expert; row r of the sum
// is sum_k mw[r, k] x[idx[r, k]], k < top, made on the way in (moe_sum_kernel's order).  MODE 3: as MODE 2, rounded as MODE 1 and then
// MODE 0, so that a layer's last update gives the same bits with the next layer's norm and without it (16,384 rows of 4096 in three layers
// 16.42 -> 16.28 ms, a captured step of 8 rows of 2048, three launches fewer, 258 -> 253 us).  MODE 2's rounding, of the update and norm
// within a layer, is its own. (The fused steps of the sums are spelt out, so that no compiler's choice moves them: the second square first
// but in MODE 2 of up to 1,024 columns.)
template <bool X_FIRST>
__device__ __forceinline__ float squares(const float4& v) {
  return fmaf(v.w, v.w, fmaf(v.z, v.z, X_FIRST ? fmaf(v.y, v.y, v.x * v.x) : fmaf(v.x, v.x, v.y * v.y)));
}

template <typename TO, int MODE, int NV, bool SUM = false>
__global__ __launch_bounds__(256) void group_rmsnorm_vec_kernel(const float* __restrict__ x, int ldx, const int* __restrict__ idx,
                                                                const float* __restrict__ w, void* __restrict__ y, int ldy, int n,
                                                                float eps, float woff, int w_one, const float* __restrict__ w2,
                                                                TO* __restrict__ h, int ldh, float woff2,
                                                                const float* __restrict__ mw, int top) {
  constexpr bool NEXT = MODE >= 2, X_FIRST = MODE == 2 && NV == 1;
  __shared__ float red[8];
  const int r = blockIdx.x, g = blockIdx.y;
  const float* xr = x + (size_t)(!SUM && idx != nullptr ? idx[r] : r) * ldx + (size_t)g * n;
  float* yr = reinterpret_cast<float*>(y) + (size_t)r * ldy + (size_t)g * n;
  const float* wg = w + (size_t)g * n;
  float4 v[NV], u[NV], a[NV], b[NV];
  const float one = w_one ? w[0] : 0.f;
  float ss = 0.f;
  if constexpr (SUM) {
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int k = 0; k < top; ++k) {
      const float* row = x + (size_t)idx[(size_t)r * top + k] * ldx + (size_t)g * n;
      const float f = mw[(size_t)r * top + k];
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = (threadIdx.x + 256 * i) * 4;
        if (c >= n) continue;
        const float4 e = *reinterpret_cast<const float4*>(row + c);
        v[i].x += f * e.x; v[i].y += f * e.y; v[i].z += f * e.z; v[i].w += f * e.w;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (threadIdx.x + 256 * i) * 4;
    u[i] = b[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (!SUM) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    a[i] = make_float4(one, one, one, one);
    if (c < n) {
      if constexpr (!SUM) v[i] = *reinterpret_cast<const float4*>(xr + c);
      if constexpr (MODE != 0) u[i] = *reinterpret_cast<const float4*>(yr + c);
      if (!w_one) a[i] = *reinterpret_cast<const float4*>(wg + c);
      if constexpr (NEXT) b[i] = *reinterpret_cast<const float4*>(w2 + (size_t)g * n + c);
    }
    ss += squares<X_FIRST>(v[i]);
  }
  const float rs = 1.f / sqrtf(block_sum_256(ss, red) / (float)n + eps);
  float s2 = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    v[i].x = u[i].x + v[i].x * rs * (a[i].x + woff); v[i].y = u[i].y + v[i].y * rs * (a[i].y + woff);
    v[i].z = u[i].z + v[i].z * rs * (a[i].z + woff); v[i].w = u[i].w + v[i].w * rs * (a[i].w + woff);
    if constexpr (NEXT) s2 += squares<X_FIRST>(v[i]);
  }
  float rs2 = 0.f;
  if constexpr (NEXT) rs2 = 1.f / sqrtf(block_sum_256(s2, red + 4) / (float)n + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (threadIdx.x + 256 * i) * 4;
    if (c >= n) continue;
    if constexpr (MODE != 0) *reinterpret_cast<float4*>(yr + c) = v[i];
    if constexpr (MODE != 1) {
      TO* hr = NEXT ? h + (size_t)r * ldh + (size_t)g * n : reinterpret_cast<TO*>(y) + (size_t)r * ldy + (size_t)g * n;
      float4 o = v[i];
      if constexpr (MODE == 2) {
        o.x *= rs2 * (b[i].x + woff2); o.y *= rs2 * (b[i].y + woff2); o.z *= rs2 * (b[i].z + woff2); o.w *= rs2 * (b[i].w + woff2);
      }
      if constexpr (MODE == 3) {
        o.x = o.x * rs2 * (b[i].x + woff2); o.y = o.y * rs2 * (b[i].y + woff2);
        o.z = o.z * rs2 * (b[i].z + woff2); o.w = o.w * rs2 * (b[i].w + woff2);
      }
      if constexpr (sizeof(TO) == 2) {
        const bf16_t e[4] = {f_to_bf16(o.x), f_to_bf16(o.y), f_to_bf16(o.z), f_to_bf16(o.w)};
        *reinterpret_cast<uint2*>(hr + c) = *reinterpret_cast<const uint2*>(e);
      } else {
        *reinterpret_cast<float4*>(hr + c) = o;
      }
    }
  }
}

// rows of up to 8,192 columns a group with 16-byte alignment throughout (8 bytes for bf16 outputs); false: the kernel above serves
template <typename TO, int MODE, bool SUM = false>
static bool group_rmsnorm_vec(const float* x, int ldx, const int* idx, const float* w, void* y, int ldy, int rows, int D, int groups,
                              float eps, float woff, int w_one, const float* w2, TO* h, int ldh, float woff2, hipStream_t st,
                              const float* mw = nullptr, int top = 0) {
  const int n = D / groups, ya = MODE == 0 ? 4 * (int)sizeof(TO) : 16;
  if (n % 4 || n > 8192 || ldx % 4 || ldy % 4 || ldh % 4 || (uintptr_t)x % 16 || (uintptr_t)y % ya || (!w_one && (uintptr_t)w % 16) ||
      (uintptr_t)w2 % 16 || (uintptr_t)h % (4 * sizeof(TO)))
    return false;
  dim3 grid(rows, groups);
#define GN_VEC(NV) hipLaunchKernelGGL((group_rmsnorm_vec_kernel<TO, MODE, NV, SUM>), grid, dim3(256), 0, st, x, ldx, idx, w, y, ldy, n, eps, woff, w_one, w2, h, ldh, woff2, mw, top)
  if (n <= 1024) GN_VEC(1);
  else if (n <= 2048) GN_VEC(2);
  else if (n <= 4096) GN_VEC(4);
  else GN_VEC(8);
#undef GN_VEC
  return true;
}

extern "C" int fls_seq_group_rmsnorm(const float* x, int ldx, const int* idx, const float* w, void* y, int ty, int ldy,
                                     int rows, int D, int groups, float eps, int add, float woff, int w_one, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (groups < 1 || D % groups) return -1;
  dim3 grid(rows, groups);
  hipStream_t st = (hipStream_t)s;
  if (add ? group_rmsnorm_vec<float, 1>(x, ldx, idx, w, y, ldy, rows, D, groups, eps, woff, w_one, nullptr, nullptr, 0, 0.f, st)
          : ty == 1 ? group_rmsnorm_vec<bf16_t, 0>(x, ldx, idx, w, y, ldy, rows, D, groups, eps, woff, w_one, nullptr, nullptr, 0, 0.f, st)
                    : group_rmsnorm_vec<float, 0>(x, ldx, idx, w, y, ldy, rows, D, groups, eps, woff, w_one, nullptr, nullptr, 0, 0.f, st)) {
    SEQ_LAUNCH_CHECK();
    return 0;
  }
  if (add) hipLaunchKernelGGL((group_rmsnorm_kernel<float, 1>), grid, dim3(256), 0, st, x, ldx, idx, w, (float*)y, ldy, D, groups, eps, woff, w_one);
  else if (ty == 1) hipLaunchKernelGGL((group_rmsnorm_kernel<bf16_t, 0>), grid, dim3(256), 0, st, x, ldx, idx, w, (bf16_t*)y, ldy, D, groups, eps, woff, w_one);
  else hipLaunchKernelGGL((group_rmsnorm_kernel<float, 0>), grid, dim3(256), 0, st, x, ldx, idx, w, (float*)y, ldy, D, groups, eps, woff, w_one);
  SEQ_LAUNCH_CHECK();
  return 0;
}

extern "C" int fls_seq_moe_sum_add_group_rmsnorm(float* x, int ldx, const float* y, int ldy, const int* dest, const float* mw, int top,
                                                 const float* w, float woff, int rows, int D, int groups, float eps, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (groups < 1 || D % groups || top < 1) return -1;
  if (!group_rmsnorm_vec<float, 1, true>(y, ldy, dest, w, x, ldx, rows, D, groups, eps, woff, 0, nullptr, nullptr, 0, 0.f, (hipStream_t)s, mw, top))
    return SEQ_NOT_SERVED;
  SEQ_LAUNCH_CHECK();
  return 0;
}

extern "C" int fls_seq_moe_sum_add_group_rmsnorm_next(float* x, int ldx, const float* y, int ldy, const int* dest, const float* mw, int top,
                                                      const float* w, float woff, const float* w2, float woff2, void* h, int th, int ldh,
                                                      int rows, int D, int groups, float eps, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (groups < 1 || D % groups || top < 1) return -1;
  hipStream_t st = (hipStream_t)s;
  if (!(th == 1 ? group_rmsnorm_vec<bf16_t, 3, true>(y, ldy, dest, w, x, ldx, rows, D, groups, eps, woff, 0, w2, (bf16_t*)h, ldh, woff2, st, mw, top)
                : group_rmsnorm_vec<float, 3, true>(y, ldy, dest, w, x, ldx, rows, D, groups, eps, woff, 0, w2, (float*)h, ldh, woff2, st, mw, top)))
    return SEQ_NOT_SERVED;
  SEQ_LAUNCH_CHECK();
  return 0;
}

extern "C" int fls_seq_add_group_rmsnorm_next(float* x, int ldx, const float* y, int ldy, const float* w, float woff, const float* w2,
                                              float woff2, void* h, int th, int ldh, int rows, int D, int groups, float eps,
                                              int in_turn, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (groups < 1 || D % groups) return -1;
  hipStream_t st = (hipStream_t)s;
#define GN_NEXT(TO, MODE) group_rmsnorm_vec<TO, MODE>(y, ldy, nullptr, w, x, ldx, rows, D, groups, eps, woff, 0, w2, (TO*)h, ldh, woff2, st)
  if (in_turn ? (th == 1 ? GN_NEXT(bf16_t, 3) : GN_NEXT(float, 3)) : (th == 1 ? GN_NEXT(bf16_t, 2) : GN_NEXT(float, 2))) {
    SEQ_LAUNCH_CHECK();
    return 0;
  }
#undef GN_NEXT
  const int rc = fls_seq_group_rmsnorm(y, ldy, nullptr, w, x, 0, ldx, rows, D, groups, eps, 1, woff, 0, s);
  return rc ? rc : fls_seq_group_rmsnorm(x, ldx, nullptr, w2, h, th, ldh, rows, D, groups, eps, 0, woff2, 0, s);
}

// ------------------------------------------------------------------------- Dynamic Tanh norm
// y[r, c] = tanh(alpha x[row, c]) w[c] + b[c]: no statistic of the row, so the work is cut over
// (row, 1024-column piece) blocks of four columns a thread.  wb = [w; b], alpha one number on the device.
template <typename TO>
__global__ __launch_bounds__(256) void dyt_norm_kernel(const float* __restrict__ x, int ldx, const int* __restrict__ idx,
                                                       const float* __restrict__ wb, const float* __restrict__ alpha,
                                                       TO* __restrict__ y, int ldy, int D, int vec) {
  const int r = blockIdx.x;
  const float a = alpha[0];
  const float* xr = x + (size_t)(idx != nullptr ? idx[r] : r) * ldx;
  const float* w = wb;
  const float* b = wb + D;
  TO* yr = y + (size_t)r * ldy;
  const int c0 = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (c0 >= D) return;
  if (vec) {
    const float4 v = *reinterpret_cast<const float4*>(xr + c0);
    const float4 wv = *reinterpret_cast<const float4*>(w + c0), bv = *reinterpret_cast<const float4*>(b + c0);
    const float o0 = tanhf(a * v.x) * wv.x + bv.x, o1 = tanhf(a * v.y) * wv.y + bv.y;
    const float o2 = tanhf(a * v.z) * wv.z + bv.z, o3 = tanhf(a * v.w) * wv.w + bv.w;
    if constexpr (sizeof(TO) == 2) {
      bf16_t e[4] = {f_to_bf16(o0), f_to_bf16(o1), f_to_bf16(o2), f_to_bf16(o3)};
      *reinterpret_cast<uint2*>(yr + c0) = *reinterpret_cast<const uint2*>(e);
    } else {
      *reinterpret_cast<float4*>(yr + c0) = make_float4(o0, o1, o2, o3);
    }
  } else {
    for (int c = c0; c < min(D, c0 + 4); ++c) stf(yr, c, tanhf(a * xr[c]) * w[c] + b[c]);
  }
}

extern "C" int fls_seq_dyt_norm(const float* x, int ldx, const int* idx, const float* wb, const float* alpha, void* y, int ty,
                                int ldy, int rows, int D, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (D < 1) return -1;
  const int vec = D % 4 == 0 && ldx % 4 == 0 && ldy % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)wb % 16 == 0 &&
                  (uintptr_t)y % 16 == 0;
  dim3 grid(rows, (D + 1023) / 1024);
  hipStream_t st = (hipStream_t)s;
  if (ty == 1) hipLaunchKernelGGL((dyt_norm_kernel<bf16_t>), grid, dim3(256), 0, st, x, ldx, idx, wb, alpha, (bf16_t*)y, ldy, D, vec);
  else hipLaunchKernelGGL((dyt_norm_kernel<float>), grid, dim3(256), 0, st, x, ldx, idx, wb, alpha, (float*)y, ldy, D, vec);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// x[r, c] += mult * y[r, c]: a sublayer's output joins the residual stream scaled
__global__ __launch_bounds__(256) void add_scaled_kernel(float* __restrict__ x, int ldx, const float* __restrict__ y, int ldy, int D,
                                                         float mult, int vec) {
  float* xr = x + (size_t)blockIdx.x * ldx;
  const float* yr = y + (size_t)blockIdx.x * ldy;
  const int c0 = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (c0 >= D) return;
  if (vec) {
    float4 a = *reinterpret_cast<const float4*>(xr + c0);
    const float4 b = *reinterpret_cast<const float4*>(yr + c0);
    a.x += mult * b.x; a.y += mult * b.y; a.z += mult * b.z; a.w += mult * b.w;
    *reinterpret_cast<float4*>(xr + c0) = a;
  } else {
    for (int c = c0; c < min(D, c0 + 4); ++c) xr[c] += mult * yr[c];
  }
}

extern "C" int fls_seq_add_scaled(float* x, int ldx, const float* y, int ldy, int rows, int D, float mult, fls_stream_t s) {
  if (rows <= 0) return 0;
  const int vec = D % 4 == 0 && ldx % 4 == 0 && ldy % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)y % 16 == 0;
  hipLaunchKernelGGL(add_scaled_kernel, dim3(rows, (D + 1023) / 1024), dim3(256), 0, (hipStream_t)s, x, ldx, y, ldy, D, mult, vec);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// x[r, c] += mult * y[r, c] and h[r, c] = tanh(alpha x[r, c]) w[c] + b[c] of the new x: the residual update and the
// next sublayer's Dynamic Tanh norm in one pass over the stream
template <typename TO>
__global__ __launch_bounds__(256) void add_scaled_dyt_kernel(float* __restrict__ x, int ldx, const float* __restrict__ y, int ldy,
                                                             float mult, const float* __restrict__ wb,
                                                             const float* __restrict__ alpha, TO* __restrict__ h, int ldh,
                                                             int D, int vec) {
  const float a = alpha[0];
  float* xr = x + (size_t)blockIdx.x * ldx;
  const float* yr = y + (size_t)blockIdx.x * ldy;
  TO* hr = h + (size_t)blockIdx.x * ldh;
  const float* w = wb;
  const float* b = wb + D;
  const int c0 = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (c0 >= D) return;
  if (vec) {
    float4 v = *reinterpret_cast<const float4*>(xr + c0);
    const float4 u = *reinterpret_cast<const float4*>(yr + c0);
    v.x += mult * u.x; v.y += mult * u.y; v.z += mult * u.z; v.w += mult * u.w;
    *reinterpret_cast<float4*>(xr + c0) = v;
    const float4 wv = *reinterpret_cast<const float4*>(w + c0), bv = *reinterpret_cast<const float4*>(b + c0);
    const float o0 = tanhf(a * v.x) * wv.x + bv.x, o1 = tanhf(a * v.y) * wv.y + bv.y;
    const float o2 = tanhf(a * v.z) * wv.z + bv.z, o3 = tanhf(a * v.w) * wv.w + bv.w;
    if constexpr (sizeof(TO) == 2) {
      bf16_t e[4] = {f_to_bf16(o0), f_to_bf16(o1), f_to_bf16(o2), f_to_bf16(o3)};
      *reinterpret_cast<uint2*>(hr + c0) = *reinterpret_cast<const uint2*>(e);
    } else {
      *reinterpret_cast<float4*>(hr + c0) = make_float4(o0, o1, o2, o3);
    }
  } else {
    for (int c = c0; c < min(D, c0 + 4); ++c) {
      const float v = xr[c] + mult * yr[c];
      xr[c] = v;
      stf(hr, c, tanhf(a * v) * w[c] + b[c]);
    }
  }
}

extern "C" int fls_seq_add_scaled_dyt(float* x, int ldx, const float* y, int ldy, float mult, const float* wb, const float* alpha,
                                      void* h, int th, int ldh, int rows, int D, fls_stream_t s) {
  if (rows <= 0) return 0;
  const int vec = D % 4 == 0 && ldx % 4 == 0 && ldy % 4 == 0 && ldh % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)y % 16 == 0 &&
                  (uintptr_t)wb % 16 == 0 && (uintptr_t)h % 16 == 0;
  dim3 grid(rows, (D + 1023) / 1024);
  hipStream_t st = (hipStream_t)s;
  if (th == 1) hipLaunchKernelGGL((add_scaled_dyt_kernel<bf16_t>), grid, dim3(256), 0, st, x, ldx, y, ldy, mult, wb, alpha, (bf16_t*)h, ldh, D, vec);
  else hipLaunchKernelGGL((add_scaled_dyt_kernel<float>), grid, dim3(256), 0, st, x, ldx, y, ldy, mult, wb, alpha, (float*)h, ldh, D, vec);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------------------- embedding
// (four columns a lane and four of its pieces' loads in flight where the rows allow it: single columns took
// a load, a wait and a store for each 256: us, 8 rows of 2,048 in bf16 2.5 -> 2.1, of 4,096 3.5 -> 2.2, 1,024 of 4,096 9.1 -> 5.9, 9,000
// 64.7 -> 35.8)
template <typename T, int VE>
__global__ __launch_bounds__(256) void embed_kernel(const int* __restrict__ ids, const T* __restrict__ table, float* __restrict__ out, int D, int V, float scale) {
  const int t = blockIdx.x;
  int id = ids[t];
  id = id < 0 ? 0 : (id >= V ? V - 1 : id);
  const T* row = table + (size_t)id * D;
  float* o = out + (size_t)t * D;
  for (int c0 = VE * threadIdx.x; c0 < D; c0 += 4 * 256 * VE) {
    RowVec<VE> v[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = row_load<VE>(row + min(c0 + x * 256 * VE, D - VE));
#pragma unroll
    for (int x = 0; x < 4; ++x) {
#pragma unroll
      for (int e = 0; e < VE; ++e) v[x].v[e] *= scale;
      if (c0 + x * 256 * VE < D) row_store<VE>(o + c0 + x * 256 * VE, v[x]);
    }
  }
}

extern "C" int fls_seq_embed(const int* ids, const void* table, int tt, float* out, int T, int D, int V, float scale, fls_stream_t s) {
  if (T <= 0 || D <= 0) return 0;
  const bool vec = D % 4 == 0 && (((uintptr_t)table | (uintptr_t)out) & 15) == 0;
#define EMBED(TT, VE) hipLaunchKernelGGL((embed_kernel<TT, VE>), dim3(T), dim3(256), 0, (hipStream_t)s, ids, (const TT*)table, out, D, V, scale)
  if (tt == 1) { if (vec) EMBED(bf16_t, 4); else EMBED(bf16_t, 1); }
  else { if (vec) EMBED(float, 4); else EMBED(float, 1); }
#undef EMBED
  SEQ_LAUNCH_CHECK();
  return 0;
}

// (V: 16 bytes where rows and strides are multiples of them, else an element)
template <typename V>
__global__ void gather_rows_kernel(const V* __restrict__ x, int ldx, const int* __restrict__ idx, V* __restrict__ y, int ldy, int D) {
  const V* xr = x + (size_t)idx[blockIdx.x] * ldx;
  V* yr = y + (size_t)blockIdx.x * ldy;
  for (int c = threadIdx.x; c < D; c += blockDim.x) yr[c] = xr[c];
}

extern "C" int fls_seq_gather_rows(const void* x, int tx, int ldx, const int* idx, void* y, int ldy, int rows, int D,
                                   fls_stream_t s) {
  if (rows <= 0) return 0;
  const int per = tx == 1 ? 8 : 4;
  // (us, bf16: 9,000 rows of 2,048 23.3 -> 12.9, of 576 10.1 -> 5.0)
  if (D % per == 0 && ldx % per == 0 && ldy % per == 0 && (((uintptr_t)x | (uintptr_t)y) & 15) == 0)
    hipLaunchKernelGGL((gather_rows_kernel<uint4>), dim3(rows), dim3(D / per <= 64 ? 64 : D / per <= 128 ? 128 : 256), 0, (hipStream_t)s, (const uint4*)x, ldx / per, idx, (uint4*)y, ldy / per, D / per);
  else if (tx == 1) hipLaunchKernelGGL((gather_rows_kernel<bf16_t>), dim3(rows), dim3(256), 0, (hipStream_t)s, (const bf16_t*)x, ldx, idx, (bf16_t*)y, ldy, D);
  else hipLaunchKernelGGL((gather_rows_kernel<float>), dim3(rows), dim3(256), 0, (hipStream_t)s, (const float*)x, ldx, idx, (float*)y, ldy, D);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// --------------------------------------------------------------------- activations between GEMMs
template <typename TO>
__global__ void xielu_kernel(const float* __restrict__ z, int ldz, const float* __restrict__ act, TO* __restrict__ y, int ldy, int cols) {
  const float ap = softplus_f(act[0]), an = 0.5f + softplus_f(act[1]);
  const float* zr = z + (size_t)blockIdx.x * ldz;
  TO* yr = y + (size_t)blockIdx.x * ldy;
  for (int c = threadIdx.x; c < cols; c += blockDim.x) {
    const float v = zr[c];
    stf(yr, c, v > 0.f ? ap * v * v + 0.5f * v : an * expm1_less_z(v) + 0.5f * v);
  }
}

extern "C" int fls_seq_xielu(const float* z, int ldz, const float* act, void* y, int ty, int ldy, int rows, int cols, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (ty == 1) hipLaunchKernelGGL((xielu_kernel<bf16_t>), dim3(rows), dim3(256), 0, (hipStream_t)s, z, ldz, act, (bf16_t*)y, ldy, cols);
  else hipLaunchKernelGGL((xielu_kernel<float>), dim3(rows), dim3(256), 0, (hipStream_t)s, z, ldz, act, (float*)y, ldy, cols);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// y = act(gate) * up for rows [gate | up]; act: 0 = silu, 1 = gelu (tanh form), 2 = clamped: g = min(gate, limit),
// u = clamp(up, -limit, limit), y = g sigmoid(alpha g) (u + 1)
template <typename TO, int ACT>
__global__ __launch_bounds__(256) void gate_mul_kernel(const float* __restrict__ gu, int ldg, TO* __restrict__ y, int ldy, int cols,
                                                       float limit, float alpha) {
  const float* gr = gu + (size_t)blockIdx.x * ldg;
  TO* yr = y + (size_t)blockIdx.x * ldy;
  for (int c = threadIdx.x; c < cols; c += blockDim.x) {
    if constexpr (ACT == 2) {
      const float g = fminf(gr[c], limit), u = fminf(fmaxf(gr[cols + c], -limit), limit);
      stf(yr, c, g / (1.f + expf(-alpha * g)) * (u + 1.f));
    } else {
      stf(yr, c, (ACT == 1 ? gelu_tanh_f(gr[c]) : silu_f(gr[c])) * gr[cols + c]);
    }
  }
}

extern "C" int fls_seq_gate_mul(const float* gu, int ldg, void* y, int ty, int ldy, int rows, int cols, int act, float limit,
                                float alpha, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (act < 0 || act > 2) return -1;
  hipStream_t st = (hipStream_t)s;
#define GATE_MUL(TO, ACT) hipLaunchKernelGGL((gate_mul_kernel<TO, ACT>), dim3(rows), dim3(256), 0, st, gu, ldg, (TO*)y, ldy, cols, limit, alpha)
  if (ty == 1) { if (act == 0) GATE_MUL(bf16_t, 0); else if (act == 1) GATE_MUL(bf16_t, 1); else GATE_MUL(bf16_t, 2); }
  else { if (act == 0) GATE_MUL(float, 0); else if (act == 1) GATE_MUL(float, 1); else GATE_MUL(float, 2); }
#undef GATE_MUL
  SEQ_LAUNCH_CHECK();
  return 0;
}

// y = f(z) elementwise; kind: 0 = tanh, 1 = gelu in its exact form 0.5 z (1 + erf(z / sqrt 2)), 2 = z itself (a cast)
template <typename TO>
__global__ void unary_kernel(const float* __restrict__ z, int ldz, TO* __restrict__ y, int ldy, int cols, int kind) {
  const float* zr = z + (size_t)blockIdx.x * ldz;
  TO* yr = y + (size_t)blockIdx.x * ldy;
  if (kind == 1) {
    for (int c = threadIdx.x; c < cols; c += blockDim.x) { const float v = zr[c]; stf(yr, c, 0.5f * v * (1.f + erff(v * 0.70710678118654752f))); }
    return;
  }
  for (int c = threadIdx.x; c < cols; c += blockDim.x) stf(yr, c, tanhf(zr[c]));
}

template <typename TO>
__global__ __launch_bounds__(256) void cast_kernel(const float* __restrict__ z, int ldz, TO* __restrict__ y, int ldy, int cols, int vec) {
  const float* zr = z + (size_t)blockIdx.x * ldz;
  TO* yr = y + (size_t)blockIdx.x * ldy;
  const int c0 = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (c0 >= cols) return;
  if (vec) {
    const float4 v = *reinterpret_cast<const float4*>(zr + c0);
    if constexpr (sizeof(TO) == 2) {
      const bf16_t e[4] = {f_to_bf16(v.x), f_to_bf16(v.y), f_to_bf16(v.z), f_to_bf16(v.w)};
      *reinterpret_cast<uint2*>(yr + c0) = *reinterpret_cast<const uint2*>(e);
    } else {
      *reinterpret_cast<float4*>(yr + c0) = v;
    }
  } else {
    for (int c = c0; c < min(cols, c0 + 4); ++c) stf(yr, c, zr[c]);
  }
}

extern "C" int fls_seq_unary(const float* z, int ldz, void* y, int ty, int ldy, int rows, int cols, int kind, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (kind < 0 || kind > 2) return -1;
  if (kind == 2) {
    const int vec = cols % 4 == 0 && ldz % 4 == 0 && ldy % 4 == 0 && (uintptr_t)z % 16 == 0 && (uintptr_t)y % 16 == 0;
    dim3 grid(rows, (cols + 1023) / 1024);
    if (ty == 1) hipLaunchKernelGGL((cast_kernel<bf16_t>), grid, dim3(256), 0, (hipStream_t)s, z, ldz, (bf16_t*)y, ldy, cols, vec);
    else hipLaunchKernelGGL((cast_kernel<float>), grid, dim3(256), 0, (hipStream_t)s, z, ldz, (float*)y, ldy, cols, vec);
    SEQ_LAUNCH_CHECK();
    return 0;
  }
  if (ty == 1) hipLaunchKernelGGL((unary_kernel<bf16_t>), dim3(rows), dim3(256), 0, (hipStream_t)s, z, ldz, (bf16_t*)y, ldy, cols, kind);
  else hipLaunchKernelGGL((unary_kernel<float>), dim3(rows), dim3(256), 0, (hipStream_t)s, z, ldz, (float*)y, ldy, cols, kind);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// first index of the row maximum.  Few rows (decoding): a block per row, so what bounds it is one block's chain of loads: 1024
// threads with 16-byte loads (32000 columns: 8 loads deep, 6 us; 256 threads of single loads 21)
#define ARGMAX_THREADS 1024
// (HOST 1: the indexes go to the address in `cell` too, 2: the rows before them as well; kernels of their own, because the question in the
// loop cost 1.6 of 15 us at 151,936 columns)
template <int HOST>
__global__ __launch_bounds__(ARGMAX_THREADS) void argmax_kernel(const float* __restrict__ z, int ldz, int cols, int vec, int* __restrict__ out,
                                                               void* const* __restrict__ cell) {
  __shared__ float bv[ARGMAX_THREADS];
  __shared__ int bi[ARGMAX_THREADS];
  const float* zr = z + (size_t)blockIdx.x * ldz;
  void* const host = HOST ? *cell : nullptr;
  float* const hr = HOST == 2 && host != nullptr ? reinterpret_cast<float*>(host) + (size_t)blockIdx.x * cols : nullptr;
  float best = -INFINITY;
  int at = 0x7fffffff;
  const int c4 = vec ? cols & ~3 : 0;
  for (int c = 4 * threadIdx.x; c < c4; c += 4 * ARGMAX_THREADS) {
    const float4 q = *reinterpret_cast<const float4*>(zr + c);
    const float v[4] = {q.x, q.y, q.z, q.w};
    if (HOST == 2 && hr != nullptr) {
      if (cols % 4 == 0) *reinterpret_cast<float4*>(hr + c) = q;
      else
#pragma unroll
        for (int i = 0; i < 4; ++i) hr[c + i] = v[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (v[i] > best || (v[i] == best && c + i < at)) { best = v[i]; at = c + i; }
  }
  for (int c = c4 + threadIdx.x; c < cols; c += ARGMAX_THREADS) {
    const float v = zr[c];
    if (HOST == 2 && hr != nullptr) hr[c] = v;
    if (v > best || (v == best && c < at)) { best = v; at = c; }
  }
  bv[threadIdx.x] = best;
  bi[threadIdx.x] = at;
  __syncthreads();
  for (int o = ARGMAX_THREADS / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      const float v = bv[threadIdx.x + o];
      const int i = bi[threadIdx.x + o];
      if (v > bv[threadIdx.x] || (v == bv[threadIdx.x] && i < bi[threadIdx.x])) { bv[threadIdx.x] = v; bi[threadIdx.x] = i; }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const int best_at = bi[0] == 0x7fffffff ? 0 : bi[0];
    out[blockIdx.x] = best_at;
    if (HOST && host != nullptr) reinterpret_cast<int*>(host)[(size_t)gridDim.x * cols + blockIdx.x] = best_at;
  }
}

extern "C" int fls_seq_argmax(const float* z, int ldz, int rows, int cols, int* out, void* const* host, int with_rows, fls_stream_t s) {
  if (rows <= 0) return 0;
  const int vec = (uintptr_t)z % 16 == 0 && ldz % 4 == 0;
  const auto kernel = host == nullptr ? argmax_kernel<0> : with_rows ? argmax_kernel<2> : argmax_kernel<1>;
  hipLaunchKernelGGL(kernel, dim3(rows), dim3(ARGMAX_THREADS), 0, (hipStream_t)s, z, ldz, cols, vec, out, host);
  SEQ_LAUNCH_CHECK();
  return 0;
}

__global__ __launch_bounds__(1024) void copy_words_kernel(const int* __restrict__ src, int* __restrict__ dst, int n) {
  const int i = 4 * (blockIdx.x * 1024 + threadIdx.x);
  if (i + 4 <= n) *reinterpret_cast<int4*>(dst + i) = *reinterpret_cast<const int4*>(src + i);
  else
    for (int j = i; j < n; ++j) dst[j] = src[j];
}

// A decode step's index arrays (some KB) over the host link by a kernel of the step's graph: 4 us, where a copy before the graph took 5
// and left 20 of idle GPU between the two (8 requests, one step of 650 us).
extern "C" int fls_seq_copy_words(const int* src, int* dst, int n, fls_stream_t s) {
  if (n <= 0) return 0;
  if ((uintptr_t)src % 16 || (uintptr_t)dst % 16) return -1;
  hipLaunchKernelGGL(copy_words_kernel, dim3((n + 4095) / 4096), dim3(1024), 0, (hipStream_t)s, src, dst, n);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------- K/V store with the key norm
template <typename TC>
__global__ __launch_bounds__(256) void kv_store_kernel(const float* __restrict__ k, int ldk, const float* __restrict__ kn, float eps,
                                                       const float* __restrict__ v, int ldv, TC* __restrict__ kc, TC* __restrict__ vc,
                                                       const int* __restrict__ kv_slot, int kcols, int vcols) {
  __shared__ float red[4];
  const int r = blockIdx.x;
  const float* kr = k + (size_t)r * ldk;
  float ss = 0.f;
  for (int c = threadIdx.x; c < kcols; c += 256) { const float x = kr[c]; ss += x * x; }
  ss = block_sum_256(ss, red);
  const float rs = 1.f / sqrtf(ss / (float)kcols + eps);
  const size_t dst = (size_t)kv_slot[r];
  for (int c = threadIdx.x; c < kcols; c += 256) stf(kc + dst * kcols, c, kr[c] * rs * kn[c]);
  const float* vr = v + (size_t)r * ldv;
  for (int c = threadIdx.x; c < vcols; c += 256) stf(vc + dst * vcols, c, vr[c]);
}

extern "C" int fls_seq_kv_store(const float* k, int ldk, const float* kn, float eps, const float* v, int ldv, void* kc, void* vc,
                                int tc, const int* kv_slot, int rows, int kcols, int vcols, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (tc == 1) hipLaunchKernelGGL((kv_store_kernel<bf16_t>), dim3(rows), dim3(256), 0, (hipStream_t)s, k, ldk, kn, eps, v, ldv, (bf16_t*)kc, (bf16_t*)vc, kv_slot, kcols, vcols);
  else hipLaunchKernelGGL((kv_store_kernel<float>), dim3(rows), dim3(256), 0, (hipStream_t)s, k, ldk, kn, eps, v, ldv, (float*)kc, (float*)vc, kv_slot, kcols, vcols);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------- per-head norm, rotation and placement
// One wave per (row, head): the head's n entries x[t, x_col + h x_hs ...] are RMS-normed over n (when w
// is given: times w[n], one weight for all heads), their first `rot` entries rotated in pairs
// (2i, 2i + 1) by the angle pos[t] * freqs[i] (fp32 angle, full-range sin / cos), and written to
// out[row, out_col + h out_hs ...] with row = row_map ? row_map[t] : t -- a matrix of rows or a page
// pool.  raw (optional, laid out like out) receives the entries as they came.  n <= 512.
#define HNR_MAX_E 8
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void head_norm_rope_kernel(const TI* x, int ldx, int x_col, int x_hs, int heads, int n,
                                                             const float* __restrict__ w, float eps,
                                                             const float* __restrict__ freqs, int rot,
                                                             const int* __restrict__ tok_pos, const int* __restrict__ row_map,
                                                             TO* out, int ldo, int out_col, int out_hs, TO* raw, int ldr,
                                                             int items, int unit_after, int half, float amp) {
  const int lane = threadIdx.x & 63;
  const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= items) return;
  const int t = item / heads, h = item % heads;
  const TI* xr = x + (size_t)t * ldx + x_col + (size_t)h * x_hs;
  float v[HNR_MAX_E];
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < HNR_MAX_E; ++e) {
    const int c = lane + 64 * e;
    v[e] = c < n ? ldf(xr, c) : 0.f;
    ss += v[e] * v[e];
  }
  const size_t row = row_map != nullptr ? (size_t)row_map[t] : (size_t)t;
  if (raw != nullptr) {
    TO* rr = raw + row * ldr + out_col + (size_t)h * out_hs;
#pragma unroll
    for (int e = 0; e < HNR_MAX_E; ++e) { const int c = lane + 64 * e; if (c < n) stf(rr, c, v[e]); }
  }
  float rs_w = 1.f;
  if (w != nullptr) {
    const float rs = 1.f / sqrtf(wave_sum(ss) / (float)n + eps);
    rs_w = rs;
#pragma unroll
    for (int e = 0; e < HNR_MAX_E; ++e) { const int c = lane + 64 * e; if (c < n) v[e] *= rs * w[c]; }
  }
  const float pos = rot > 0 ? (float)tok_pos[t] : 0.f;
  TO* orow = out + row * ldo + out_col + (size_t)h * out_hs;
  // the pair's other entry: in the neighbouring lane for pairs (2i, 2i + 1); for pairs (i, i + rot / 2) it is read
  // from the row again and normed alike (all of them before anything is stored: out may be x)
  float oth[HNR_MAX_E];
  const int hr = rot >> 1;
#pragma unroll
  for (int e = 0; e < HNR_MAX_E; ++e) {
    const int c = lane + 64 * e;
    oth[e] = __shfl_xor(v[e], 1, 64);
    if (half && c < rot) {
      const int pc = c >= hr ? c - hr : c + hr;
      oth[e] = ldf(xr, pc) * (w != nullptr ? rs_w * w[pc] : 1.f);
    }
  }
#pragma unroll
  for (int e = 0; e < HNR_MAX_E; ++e) {
    const int c = lane + 64 * e;
    float val = v[e];
    if (c < rot) {
      const bool second = half ? c >= hr : (c & 1);
      const int fi = half ? (second ? c - hr : c) : (c >> 1);
      const float ang = pos * freqs[fi];
      const float cs = amp * cosf(ang), sn = amp * sinf(ang);
      val = second ? v[e] * cs + oth[e] * sn : v[e] * cs - oth[e] * sn;
    }
    if (!unit_after) { if (c < n) stf(orow, c, val); }
    else v[e] = val;
  }
  if (unit_after) {                                  // (block-uniform)
    float s2 = 0.f;
#pragma unroll
    for (int e = 0; e < HNR_MAX_E; ++e) s2 += v[e] * v[e];          // (entries past n are zeros)
    const float rs = 1.f / sqrtf(wave_sum(s2) / (float)n + eps);
#pragma unroll
    for (int e = 0; e < HNR_MAX_E; ++e) { const int c = lane + 64 * e; if (c < n) stf(orow, c, v[e] * rs); }
  }
}

// The same for heads of whole vectors of four entries, n <= 256 EV (four or eight entries a lane): a head takes 2^shift lanes, a block
// `rb` rows with all their heads, or, where that would be few blocks, hb heads of a row.  The general kernel above works every head's
// angles out anew, sine and cosine of each entry of each pair, and that, not memory, bounds it; here a block makes a row's table once,
// in LDS, and its loads and stores are 16 bytes a lane.
// 6,700 rows of 16 heads of 128, all turned, fp32 in place 64 -> 22 us (110 MB: 23 at the rate of a copy), of 64 42 -> 12; 9,700 of 16 x 128
// in bf16 79 -> 23; 6,700 of one head of 512, normed, 9.3 -> 7.9.
template <typename TI, typename TO, int EV>
__global__ __launch_bounds__(256) void head_norm_rope_rows(const TI* x, int ldx, int x_col, int x_hs, int heads, int n,
                                                           const float* __restrict__ w, float eps, const float* __restrict__ freqs, int rot,
                                                           const int* __restrict__ tok_pos, const int* __restrict__ row_map, TO* out, int ldo,
                                                           int out_col, int out_hs, TO* raw, int ldr, int rows, int unit_after, int half,
                                                           float amp, int shift, int rb, int hb) {
  __shared__ float2 turn[1024];                              // (rb rows of rot / 2 angles: 128 n / 2^shift at most)
  const int t0 = blockIdx.x * rb, hr = rot >> 1, h0 = blockIdx.y * hb, nh = min(hb, heads - h0);
  if (rot > 0) {
    for (int i = threadIdx.x; i < rb * hr; i += 256) {
      const int r = i / hr;
      if (t0 + r < rows) {
        const float ang = (float)tok_pos[t0 + r] * freqs[i - r * hr];
        turn[i] = make_float2(amp * cosf(ang), amp * sinf(ang));
      }
    }
    __syncthreads();
  }
  const int lanes = 1 << shift, sub = threadIdx.x & (lanes - 1), base = (threadIdx.x & 63) - sub;
  for (int it = threadIdx.x >> shift; it < rb * nh; it += 256 >> shift) {          // (a head's lanes together)
    const int r = it / nh, h = h0 + it - r * nh, t = t0 + r;
    if (t >= rows) break;
    const TI* xr = x + (size_t)t * ldx + x_col + (size_t)h * x_hs;
    RowVec<4> v[EV];
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < EV; ++e) {
      const int c = 4 * (sub + (e << shift));
      v[e] = c < n ? row_load<4>(xr + c) : RowVec<4>{};
#pragma unroll
      for (int j = 0; j < 4; ++j) ss += v[e].v[j] * v[e].v[j];
    }
    const size_t row = row_map != nullptr ? (size_t)row_map[t] : (size_t)t;
    if (raw != nullptr) {
      TO* rr = raw + row * ldr + out_col + (size_t)h * out_hs;
#pragma unroll
      for (int e = 0; e < EV; ++e) { const int c = 4 * (sub + (e << shift)); if (c < n) row_store<4>(rr + c, v[e]); }
    }
    if (w != nullptr) {
      for (int o = 1; o < lanes; o <<= 1) ss += __shfl_xor(ss, o, 64);
      const float rs = 1.f / sqrtf(ss / (float)n + eps);
#pragma unroll
      for (int e = 0; e < EV; ++e) {
        const int c = 4 * (sub + (e << shift));
        if (c < n) {
          const float4 wc = *reinterpret_cast<const float4*>(w + c);
          v[e].v[0] *= rs * wc.x; v[e].v[1] *= rs * wc.y; v[e].v[2] *= rs * wc.z; v[e].v[3] *= rs * wc.w;
        }
      }
    }
    if (rot > 0) {
      const float2* tr = turn + r * hr;
      float oth[EV][4];
      if (half) {                                            // the pair's other entry: another lane's, of whichever of its vectors
#pragma unroll
        for (int e = 0; e < EV; ++e) {
          const int c = 4 * (sub + (e << shift)), pc = c >= rot ? c : c >= hr ? c - hr : c + hr, q = pc >> 2;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            oth[e][j] = __shfl(v[0].v[j], base + (q & (lanes - 1)), 64);
            if constexpr (EV == 2) {
              const float far = __shfl(v[1].v[j], base + (q & (lanes - 1)), 64);
              if (q >> shift) oth[e][j] = far;
            }
          }
        }
      }
#pragma unroll
      for (int e = 0; e < EV; ++e) {
        const int c = 4 * (sub + (e << shift));
        if (c >= rot) continue;
        if (half) {
          const bool second = c >= hr;
          const float2* f = tr + (second ? c - hr : c);
#pragma unroll
          for (int j = 0; j < 4; ++j) v[e].v[j] = second ? v[e].v[j] * f[j].x + oth[e][j] * f[j].y : v[e].v[j] * f[j].x - oth[e][j] * f[j].y;
        } else {
          const float2* f = tr + (c >> 1);
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const float a = v[e].v[2 * j], b = v[e].v[2 * j + 1];
            v[e].v[2 * j] = a * f[j].x - b * f[j].y;
            v[e].v[2 * j + 1] = b * f[j].x + a * f[j].y;
          }
        }
      }
    }
    if (unit_after) {
      float s2 = 0.f;
#pragma unroll
      for (int e = 0; e < EV; ++e)
#pragma unroll
        for (int j = 0; j < 4; ++j) s2 += v[e].v[j] * v[e].v[j];
      for (int o = 1; o < lanes; o <<= 1) s2 += __shfl_xor(s2, o, 64);
      const float rs = 1.f / sqrtf(s2 / (float)n + eps);
#pragma unroll
      for (int e = 0; e < EV; ++e)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[e].v[j] *= rs;
    }
    TO* orow = out + row * ldo + out_col + (size_t)h * out_hs;
#pragma unroll
    for (int e = 0; e < EV; ++e) { const int c = 4 * (sub + (e << shift)); if (c < n) row_store<4>(orow + c, v[e]); }
  }
}

// rows of elements of `size` bytes, heads `hs` apart from column `col` on: vectors of four all aligned?
static bool vectors_of_four(const void* p, int size, int ld, int col, int hs, int heads) {
  return (uintptr_t)p % (4 * size) == 0 && ld % 4 == 0 && col % 4 == 0 && (heads == 1 || hs % 4 == 0);
}

extern "C" int fls_seq_head_norm_rope(const void* x, int tx, int ldx, int x_col, int x_hs, int heads, int n, const float* w,
                                      float eps, const float* freqs, int rot, const int* tok_pos, const int* row_map, void* out,
                                      int to, int ldo, int out_col, int out_hs, void* raw, int ldr, int rows, int unit_after,
                                      int half, float amp, fls_stream_t s) {
  if (rows <= 0 || heads <= 0) return 0;
  if (n < 1 || n > 64 * HNR_MAX_E || rot < 0 || rot > n || (rot & 1) || (rot > 0 && (freqs == nullptr || tok_pos == nullptr))) return -1;
  const int items = rows * heads;
  dim3 grid((items + 3) / 4);
  hipStream_t st = (hipStream_t)s;
  const int si = tx == 1 ? 2 : 4, so = to == 1 ? 2 : 4;
  if (n % 4 == 0 && rot % (half ? 8 : 4) == 0 && vectors_of_four(x, si, ldx, x_col, x_hs, heads) &&
      vectors_of_four(out, so, ldo, out_col, out_hs, heads) && (raw == nullptr || vectors_of_four(raw, so, ldr, out_col, out_hs, heads)) &&
      (w == nullptr || (uintptr_t)w % 16 == 0)) {
    int shift = 0;
    while ((4 << shift) < n && shift < 6) ++shift;
    const int per = heads << shift, rb = per >= 256 ? 1 : 256 / per, side = 256 >> shift;       // (heads that a block has side by side)
    const int parts = per <= 256 || rows >= 1024 ? 1 : min((heads + side - 1) / side, (1024 + rows - 1) / rows), hb = (heads + parts - 1) / parts;
    const dim3 blocks((rows + rb - 1) / rb, (heads + hb - 1) / hb);
#define HNR_(TI, TO, EV) hipLaunchKernelGGL((head_norm_rope_rows<TI, TO, EV>), blocks, dim3(256), 0, st, (const TI*)x, ldx, x_col, x_hs, heads, n, w,  \
                                            eps, freqs, rot, tok_pos, row_map, (TO*)out, ldo, out_col, out_hs, (TO*)raw, ldr, rows, unit_after, half,  \
                                            amp, shift, rb, hb)
#define HNR(TI, TO)                  \
  do {                               \
    if (n <= 256) HNR_(TI, TO, 1);   \
    else HNR_(TI, TO, 2);            \
  } while (0)
    if (tx == 1 && to == 1) HNR(bf16_t, bf16_t);
    else if (tx == 1) HNR(bf16_t, float);
    else if (to == 1) HNR(float, bf16_t);
    else HNR(float, float);
#undef HNR
#undef HNR_
    SEQ_LAUNCH_CHECK();
    return 0;
  }
#define HNR(TI, TO) hipLaunchKernelGGL((head_norm_rope_kernel<TI, TO>), grid, dim3(256), 0, st, (const TI*)x, ldx, x_col, x_hs, heads, \
                                       n, w, eps, freqs, rot, tok_pos, row_map, (TO*)out, ldo, out_col, out_hs, (TO*)raw, ldr, items, unit_after, half, amp)
  if (tx == 1 && to == 1) HNR(bf16_t, bf16_t);
  else if (tx == 1) HNR(bf16_t, float);
  else if (to == 1) HNR(float, bf16_t);
  else HNR(float, float);
#undef HNR
  SEQ_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------------ mixture of experts
// one thread per token: the `top` largest logits are chosen (ties: the lower expert) and weighted by the softmax over the chosen
// logits only
#define MOE_MAX_TOP 16
__global__ void moe_route_kernel(const float* __restrict__ logits, int ldl, int T, int E, int top, int* __restrict__ ids,
                                 float* __restrict__ w) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  const float* l = logits + (size_t)t * ldl;
  int chosen[MOE_MAX_TOP];
  float val[MOE_MAX_TOP];
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int be = -1;
    for (int e = 0; e < E; ++e) {
      bool used = false;
      for (int j = 0; j < k; ++j) used |= (chosen[j] == e);
      if (used) continue;
      const float c = l[e];
      if (be < 0 || c > best) { best = c; be = e; }
    }
    chosen[k] = be;
    val[k] = best;
  }
  const float mx = val[0];                          // (the first choice is the largest)
  float sum = 0.f;
  for (int k = 0; k < top; ++k) { val[k] = expf(val[k] - mx); sum += val[k]; }
  const float inv = 1.f / sum;
  for (int k = 0; k < top; ++k) {
    ids[(size_t)t * top + k] = chosen[k];
    w[(size_t)t * top + k] = val[k] * inv;
  }
}

// entries per expert: a block counts its entries in LDS, then adds one number per expert to hist
#define MOE_MAX_E 1024
__global__ __launch_bounds__(256) void moe_hist_kernel(const int* __restrict__ ids, int n, int E, int* __restrict__ hist) {
  __shared__ int h[MOE_MAX_E];
  for (int e = threadIdx.x; e < E; e += 256) h[e] = 0;
  __syncthreads();
  for (int i = blockIdx.x * 4096 + threadIdx.x; i < min(n, (int)(blockIdx.x + 1) * 4096); i += 256) atomicAdd(&h[ids[i]], 1);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 256)
    if (h[e]) atomicAdd(hist + e, h[e]);
}

// one thread per token: scores sigmoid(logit); the experts form `groups` equal groups of neighbours, a group is worth the
// sum of its two largest scores, only experts of the `keep` best groups compete (ties: the lower group / expert);
// weights = score / (sum of the chosen + 1e-20) * scale.  groups <= 1: every expert competes
#define MOE_MAX_GROUPS 64
__global__ void moe_route_grouped_kernel(const float* __restrict__ logits, int ldl, int T, int E, int top, int groups, int keep,
                                         float scale, int* __restrict__ ids, float* __restrict__ w) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  const float* l = logits + (size_t)t * ldl;
  unsigned long long kept = ~0ull;
  const int per = groups > 1 ? E / groups : E;
  if (groups > 1) {
    float worth[MOE_MAX_GROUPS];
    for (int g = 0; g < groups; ++g) {
      float b1 = -1.f, b2 = -1.f;                     // (scores lie in (0, 1))
      for (int e = g * per; e < (g + 1) * per; ++e) {
        const float sc = sigmoid_f(l[e]);
        if (sc > b1) { b2 = b1; b1 = sc; } else if (sc > b2) { b2 = sc; }
      }
      worth[g] = b1 + (b2 > 0.f ? b2 : 0.f);
    }
    kept = 0ull;
    for (int k = 0; k < keep; ++k) {
      float best = -1.f;
      int bg = 0;
      for (int g = 0; g < groups; ++g)
        if (!((kept >> g) & 1ull) && worth[g] > best) { best = worth[g]; bg = g; }
      kept |= 1ull << bg;
    }
  }
  int chosen[MOE_MAX_TOP];
  float val[MOE_MAX_TOP];
  float sum = 0.f;
  for (int k = 0; k < top; ++k) {
    float best = -1.f;
    int be = 0;
    for (int e = 0; e < E; ++e) {
      if (groups > 1 && !((kept >> (e / per)) & 1ull)) continue;
      bool used = false;
      for (int j = 0; j < k; ++j) used |= (chosen[j] == e);
      if (used) continue;
      const float sc = sigmoid_f(l[e]);
      if (sc > best) { best = sc; be = e; }
    }
    chosen[k] = be;
    val[k] = best;
    sum += best;
  }
  const float inv = scale / (sum + 1e-20f);
  for (int k = 0; k < top; ++k) {
    ids[(size_t)t * top + k] = chosen[k];
    w[(size_t)t * top + k] = val[k] * inv;
  }
}

// Softmax scores with a correction for the choice, a wave per token: lane l holds experts l, l + 64, ...  Every choice is a
// maximum over the wave (ties: the lower index).  FUSED (one block, few tokens): afterwards the block counts the entries
// per expert in LDS, scans the counts and gives every entry its row, so that a decode step routes in one launch (8 rows:
// 4.5 us, 22 in five launches).  bare: the weights are the scores as they are.
#define RSG_FUSED_WAVES 16
template <int NE, int NW, bool FUSED>
__global__ __launch_bounds__(64 * NW) void moe_route_softmax_grouped_kernel(const float* __restrict__ logits, int ldl,
                                                                            const float* __restrict__ corr, int T, int E, int top,
                                                                            int groups, int keep, float scale, int bare,
                                                                            int* __restrict__ ids, float* __restrict__ w,
                                                                            int* __restrict__ hist, int* __restrict__ offs,
                                                                            int* __restrict__ dest, int* __restrict__ rows) {
  __shared__ float choice[NW][NE * 64];
  __shared__ int cnt[MOE_MAX_E], start[FUSED ? MOE_MAX_E : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int e = threadIdx.x; e < E; e += 64 * NW) cnt[e] = 0;
  __syncthreads();
  for (int t = blockIdx.x * NW + wave; t < T; t += gridDim.x * NW) {
    const float* l = logits + (size_t)t * ldl;
    float sc[NE], ch[NE];
    float mx = -INFINITY, sum = 0.f;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = lane + 64 * i;
      sc[i] = e < E ? l[e] : -INFINITY;
      mx = fmaxf(mx, sc[i]);
    }
    mx = wave_max(mx);
#pragma unroll
    for (int i = 0; i < NE; ++i) { sc[i] = lane + 64 * i < E ? expf(sc[i] - mx) : 0.f; sum += sc[i]; }
    const float inv = 1.f / wave_sum(sum);
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = lane + 64 * i;
      sc[i] *= inv;
      const float c = sc[i] + (corr != nullptr && e < E ? corr[e] : 0.f);
      ch[i] = e < E ? (c > -3e38f ? c : -3e38f) : -INFINITY;          // (an index that exists always beats one that does not)
    }
    if (groups > 1) {
#pragma unroll
      for (int i = 0; i < NE; ++i) choice[wave][lane + 64 * i] = ch[i];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const int per = E / groups;
      float worth = -INFINITY;
      if (lane < groups)
        for (int e = 0; e < per; ++e) worth = fmaxf(worth, choice[wave][lane * per + e]);
      bool open = lane < groups;
      unsigned long long kept = 0ull;
      for (int k = 0; k < keep; ++k) {
        const float best = wave_max(open ? worth : -INFINITY);
        const unsigned long long at = __ballot(open && worth == best);
        const int g = __ffsll((long long)(at ? at : __ballot(open))) - 1;
        if (lane == g) open = false;
        kept |= 1ull << g;
      }
#pragma unroll
      for (int i = 0; i < NE; ++i) {
        const int e = lane + 64 * i;
        if (e < E && !((kept >> (e / per)) & 1ull)) ch[i] = -INFINITY;
      }
      __builtin_amdgcn_wave_barrier();
    }
    int my_e = 0;
    float my_s = 0.f, total = 0.f;
    for (int k = 0; k < top; ++k) {
      float best = -INFINITY;
#pragma unroll
      for (int i = 0; i < NE; ++i) best = fmaxf(best, ch[i]);
      const float bw = wave_max(best);
      int e = 0x7fffffff;                                    // the lowest of the largest
#pragma unroll
      for (int i = NE - 1; i >= 0; --i) {
        const unsigned long long at = __ballot(ch[i] == bw && bw > -INFINITY);
        if (at != 0) e = 64 * i + __ffsll((long long)at) - 1;
      }
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < NE; ++i)
        if (lane + 64 * i == e) { s = sc[i]; ch[i] = -INFINITY; }
      s = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), e & 63));
      total += s;
      if (lane == k) { my_e = e; my_s = s; }
    }
    if (lane < top) {
      ids[(size_t)t * top + lane] = my_e;
      w[(size_t)t * top + lane] = bare ? my_s : my_s * (scale / (total + 1e-20f));
      atomicAdd(&cnt[my_e], 1);
    }
  }
  __syncthreads();
  if constexpr (!FUSED) {                            // (one number per block and expert)
    for (int e = threadIdx.x; e < E; e += 64 * NW)
      if (hist != nullptr && cnt[e]) atomicAdd(hist + e, cnt[e]);
  } else {
    if (wave == 0) {
      const int per = (E + 63) / 64, e0 = min(E, lane * per), e1 = min(E, e0 + per);
      int own = 0;
      for (int e = e0; e < e1; ++e) own += cnt[e];
      int acc = own;
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(acc, o, 64);
        if (lane >= o) acc += v;
      }
      if (lane == 63) offs[E] = acc;
      acc -= own;
      for (int e = e0; e < e1; ++e) { offs[e] = acc; start[e] = acc; acc += cnt[e]; }
    }
    __syncthreads();
    // (the block's own writes of ids: visible to it after the barrier)
    for (int i = threadIdx.x; i < T * top; i += 64 * NW) {
      const int p = atomicAdd(&start[ids[i]], 1);
      dest[i] = p;
      rows[p] = i / top;
    }
  }
}

static int moe_route_softmax(const float* logits, int ldl, const float* corr, int T, int E, int top, int groups, int keep, float scale,
                             int bare, int* ids, float* w, int* hist, int* offs, int* dest, int* rows, hipStream_t st) {
  const bool fused = T <= FLS_SEQ_ROUTE_FUSED;
  // (a block adds its counts once: 16384 tokens of 8 experts 13 us; with 4 waves a block, 1024 blocks of them 22)
#define RSG_WAVES(NE) ((NE) > 4 ? 8 : RSG_FUSED_WAVES)
#define RSG_(NE, FUSED, BLOCKS) hipLaunchKernelGGL((moe_route_softmax_grouped_kernel<NE, RSG_WAVES(NE), FUSED>), dim3(BLOCKS),        \
                                                   dim3(64 * RSG_WAVES(NE)), 0, st, logits, ldl, corr, T, E, top, groups, keep,      \
                                                   scale, bare, ids, w, hist, offs, dest, rows)
#define RSG(NE)                                                                                                                     \
  do {                                                                                                                              \
    if (fused) RSG_(NE, true, 1);                                                                                                   \
    else RSG_(NE, false, min(512, (T + RSG_WAVES(NE) - 1) / RSG_WAVES(NE)));                                                        \
  } while (0)
  if (E <= 64) RSG(1);
  else if (E <= 128) RSG(2);
  else if (E <= 256) RSG(4);
  else RSG(16);
#undef RSG
#undef RSG_
#undef RSG_WAVES
  SEQ_LAUNCH_CHECK();
  return 0;
}

extern "C" int fls_seq_moe_route_softmax_grouped(const float* logits, int ldl, const float* corr, int T, int E, int top, int groups,
                                                 int keep, float scale, int* ids, float* w, int* hist, int* offs, int* dest, int* rows,
                                                 fls_stream_t s) {
  if (T <= 0) return 0;
  if (top < 1 || top > MOE_MAX_TOP || top > E || E > MOE_MAX_E || groups < 0 || groups > MOE_MAX_GROUPS) return -1;
  if (groups > 1 && (E % groups || keep < 1 || keep > groups || keep * (E / groups) < top)) return -1;
  return moe_route_softmax(logits, ldl, corr, T, E, top, groups, keep, scale, 0, ids, w, hist, offs, dest, rows, (hipStream_t)s);
}

extern "C" int fls_seq_moe_route_grouped(const float* logits, int ldl, int T, int E, int top, int groups, int keep, float scale,
                                         int* ids, float* w, int* hist, fls_stream_t s) {
  if (T <= 0) return 0;
  if (top < 1 || top > MOE_MAX_TOP || top > E || E > MOE_MAX_E || groups < 0 || groups > MOE_MAX_GROUPS) return -1;
  if (groups > 1 && (E % groups || keep < 1 || keep > groups || keep * (E / groups) < top)) return -1;
  hipLaunchKernelGGL(moe_route_grouped_kernel, dim3((T + 127) / 128), dim3(128), 0, (hipStream_t)s, logits, ldl, T, E, top, groups,
                     keep, scale, ids, w);
  SEQ_LAUNCH_CHECK();
  if (hist != nullptr) hipLaunchKernelGGL(moe_hist_kernel, dim3((T * top + 4095) / 4096), dim3(256), 0, (hipStream_t)s, ids, T * top, E, hist);
  SEQ_LAUNCH_CHECK();
  return 0;
}

extern "C" int fls_seq_moe_route(const float* logits, int ldl, const float* corr, int T, int E, int top, int* ids, float* w,
                                 int* hist, int* offs, int* dest, int* rows, fls_stream_t s) {
  if (T <= 0) return 0;
  if (top < 1 || top > MOE_MAX_TOP || top > E || E > MOE_MAX_E) return -1;
  if (corr != nullptr) return moe_route_softmax(logits, ldl, corr, T, E, top, 0, 0, 1.f, 1, ids, w, hist, offs, dest, rows, (hipStream_t)s);
  hipLaunchKernelGGL(moe_route_kernel, dim3((T + 127) / 128), dim3(128), 0, (hipStream_t)s, logits, ldl, T, E, top, ids, w);
  SEQ_LAUNCH_CHECK();
  if (hist != nullptr) hipLaunchKernelGGL(moe_hist_kernel, dim3((T * top + 4095) / 4096), dim3(256), 0, (hipStream_t)s, ids, T * top, E, hist);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// Entries to their rows: every block scans the counts for itself (lane l of its first wave sums a run of ceil(E / 64) experts, the runs'
// starts come from a prefix sum over the lanes), the first one leaves them in offs; it ranks its entries in LDS and takes its places with
// one atomic per expert (32768 entries of 8 experts: 50 us with an atomic per wave and expert, 6.8 here).
// SELF (few entries): every block counts all of them for itself, and those of the blocks before it for its places: no counts and cursors
// that have to be zeroed first, and no atomics on memory (a launch less for each layer with experts of a prompt's portion).
#define PLACE_THREADS 1024
template <bool SELF>
__global__ __launch_bounds__(PLACE_THREADS) void moe_place_kernel(const int* __restrict__ ids, int n, int top, const int* __restrict__ hist, int E,
                                                        int* __restrict__ offs, int* __restrict__ cursor, int* __restrict__ dest,
                                                        int* __restrict__ rows) {
  __shared__ int start[MOE_MAX_E], cnt[MOE_MAX_E], tot[SELF ? MOE_MAX_E : 1], bef[SELF ? MOE_MAX_E : 1];
  for (int e = threadIdx.x; e < E; e += PLACE_THREADS) {
    cnt[e] = 0;
    if constexpr (SELF) tot[e] = bef[e] = 0;
  }
  if constexpr (SELF) {
    __syncthreads();
    for (int base = threadIdx.x & ~63; base < n; base += PLACE_THREADS) {        // 64 entries a wave; the lanes of one expert count together
      const int at = base + (threadIdx.x & 63);
      const int e = at < n ? ids[at] : -1;
      unsigned long long todo = __ballot(at < n);
      while (todo) {
        const int leader = __ffsll((long long)todo) - 1, el = __shfl(e, leader, 64);
        const unsigned long long same = __ballot(e == el);
        if ((int)(threadIdx.x & 63) == leader) {
          atomicAdd(&tot[el], __popcll(same));
          if (base < (int)blockIdx.x * PLACE_THREADS) atomicAdd(&bef[el], __popcll(same));
        }
        todo &= ~same;
      }
    }
    __syncthreads();
  }
  const auto count = [&](int e) { return SELF ? tot[SELF ? e : 0] : hist[e]; };
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x, per = (E + 63) / 64;
    const int e0 = min(E, lane * per), e1 = min(E, e0 + per);
    int own = 0;
    for (int e = e0; e < e1; ++e) own += count(e);
    int acc = own;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(acc, o, 64);
      if (lane >= o) acc += v;
    }
    const bool first = blockIdx.x == 0;
    if (first && lane == 63) offs[E] = acc;
    acc -= own;
    for (int e = e0; e < e1; ++e) {
      start[e] = acc + (SELF ? bef[SELF ? e : 0] : 0);
      if (first) offs[e] = acc;
      acc += count(e);
    }
  }
  __syncthreads();
  // the lanes of a wave that go to the same expert take their ranks in the block together: the first of them adds their number
  const int i = blockIdx.x * PLACE_THREADS + threadIdx.x;
  const bool valid = i < n;
  const int e = valid ? ids[i] : -1;
  const int lane = threadIdx.x & 63;
  int rank = 0;
  unsigned long long todo = __ballot(valid);
  while (todo) {
    const int leader = __ffsll((long long)todo) - 1;
    const int el = __shfl(e, leader, 64);
    const unsigned long long same = __ballot(valid && e == el);
    int base = 0;
    if (lane == leader) base = atomicAdd(&cnt[el], __popcll(same));
    base = __shfl(base, leader, 64);
    if (valid && e == el) rank = base + __popcll(same & ((1ull << lane) - 1ull));
    todo &= ~same;
  }
  __syncthreads();
  if constexpr (!SELF) {
    for (int g = threadIdx.x; g < E; g += PLACE_THREADS)
      if (cnt[g]) start[g] += atomicAdd(cursor + g, cnt[g]);
    __syncthreads();
  }
  if (valid) {
    const int p = start[e] + rank;
    dest[i] = p;
    rows[p] = i / top;
  }
}

extern "C" int fls_seq_moe_place(const int* ids, int n, int top, const int* hist, int E, int* offs, int* cursor, int* dest, int* rows,
                                 fls_stream_t s) {
  if (n <= 0) return 0;
  if (E < 1 || E > MOE_MAX_E) return -1;
  const dim3 blocks((n + PLACE_THREADS - 1) / PLACE_THREADS);
  if (hist == nullptr) {
    hipLaunchKernelGGL((moe_place_kernel<true>), blocks, dim3(PLACE_THREADS), 0, (hipStream_t)s, ids, n, top, hist, E, offs, cursor, dest, rows);
  } else {
    hipLaunchKernelGGL((moe_place_kernel<false>), blocks, dim3(PLACE_THREADS), 0, (hipStream_t)s, ids, n, top, hist, E, offs, cursor, dest, rows);
  }
  SEQ_LAUNCH_CHECK();
  return 0;
}

__global__ void moe_sum_kernel(const float* __restrict__ y, int ldy, const int* __restrict__ dest, const float* __restrict__ w,
                               float* __restrict__ out, int ldo, int top, int D) {
  const int t = blockIdx.x;
  for (int c = threadIdx.x; c < D; c += blockDim.x) {
    float acc = 0.f;
    for (int k = 0; k < top; ++k) acc += w[(size_t)t * top + k] * y[(size_t)dest[(size_t)t * top + k] * ldy + c];
    out[(size_t)t * ldo + c] = acc;
  }
}

extern "C" int fls_seq_moe_sum(const float* y, int ldy, const int* dest, const float* w, float* out, int ldo, int T, int top,
                               int D, fls_stream_t s) {
  if (T <= 0) return 0;
  hipLaunchKernelGGL(moe_sum_kernel, dim3(T), dim3(256), 0, (hipStream_t)s, y, ldy, dest, w, out, ldo, top, D);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// x[t, c] += mult * (sum_k w[t, k] y[dest[t, k], c] + sigmoid(gate[t]) shared[t, c]); shared / gate nullable
__global__ __launch_bounds__(256) void moe_combine_kernel(float* __restrict__ x, int ldx, const float* __restrict__ y, int ldy,
                                                          const int* __restrict__ dest, const float* __restrict__ w, int top,
                                                          const float* __restrict__ shared, int lds, const float* __restrict__ gate,
                                                          int ldg, int D, float mult) {
  const int t = blockIdx.x;
  const float sg = shared == nullptr ? 0.f : (gate != nullptr ? sigmoid_f(gate[(size_t)t * ldg]) : 1.f);
  for (int c = blockIdx.y * 256 + threadIdx.x; c < D; c += 256 * gridDim.y) {
    float acc = 0.f;
    for (int k = 0; k < top; ++k) acc += w[(size_t)t * top + k] * y[(size_t)dest[(size_t)t * top + k] * ldy + c];
    if (shared != nullptr) acc += sg * shared[(size_t)t * lds + c];
    x[(size_t)t * ldx + c] += mult * acc;
  }
}

extern "C" int fls_seq_moe_combine(float* x, int ldx, const float* y, int ldy, const int* dest, const float* w, int T, int top,
                                   const float* shared, int lds, const float* gate, int ldg, int D, float mult, fls_stream_t s) {
  if (T <= 0) return 0;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(T, (D + 1023) / 1024), dim3(256), 0, (hipStream_t)s, x, ldx, y, ldy, dest, w, top, shared,
                     lds, gate, ldg, D, mult);
  SEQ_LAUNCH_CHECK();
  return 0;
}

extern "C" int fls_seq_version(void) { return 26; }
