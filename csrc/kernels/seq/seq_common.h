// Shared device helpers of the stateful-model kernels (csrc/kernels/seq): element types and
// conversions.  Element type codes of the C API: 0 = fp32, 1 = bf16.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef uint16_t bf16_t;   // raw bfloat16 bits

__device__ __forceinline__ float bf16_to_f(bf16_t v) { return __uint_as_float(((uint32_t)v) << 16); }
__device__ __forceinline__ bf16_t f_to_bf16(float f) {          // round to nearest even
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((u >> 16) | 0x40);   // NaN stays NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float ldf(const float* p, size_t i) { return p[i]; }
__device__ __forceinline__ float ldf(const bf16_t* p, size_t i) { return bf16_to_f(p[i]); }
__device__ __forceinline__ void stf(float* p, size_t i, float v) { p[i] = v; }
__device__ __forceinline__ void stf(bf16_t* p, size_t i, float v) { p[i] = f_to_bf16(v); }

// v of another lane of this lane's row of 16, by a DPP control (no LDS)
template <int CTRL>
__device__ __forceinline__ float row_dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// sum over the 16 lanes of a row; every lane gets the result (pairs, quads, then the mirrored half and the mirrored row)
__device__ __forceinline__ float row16_sum(float v) {
  v += row_dpp<0xB1>(v);           // lanes 1 0 3 2
  v += row_dpp<0x4E>(v);           // lanes 2 3 0 1
  v += row_dpp<0x141>(v);          // mirrored within 8
  v += row_dpp<0x140>(v);          // mirrored within 16
  return v;
}
// maximum / sum over the wave, every lane gets it: the four steps within a row of 16 by DPP, the two across rows by lane swaps.  Six
// shuffles through LDS took some 400 cycles in a kernel's chain, these 60 (24 tokens routed over 10 outputs
// in 5 groups 7.9 -> 5.4 us, 64 over 64 in 8 28 -> 18)
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, row_dpp<0xB1>(v));
  v = fmaxf(v, row_dpp<0x4E>(v));
  v = fmaxf(v, row_dpp<0x141>(v));
  v = fmaxf(v, row_dpp<0x140>(v));
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float wave_sum(float v) {
  v = row16_sum(v);
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
// sum over the 256 threads of a block (red: 4 floats of LDS); every thread gets the result
__device__ __forceinline__ float block_sum_256(float v, float* red) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}
__device__ __forceinline__ float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }
// x, computed here and not in a branch of what chooses it: a lane's short alternatives side by side are cheaper than a wave's turns.  SIDES
// false: as the compiler likes (the same value).  A loop over accumulators is not unrolled with the assembly in it, and indexed ones go to
// scratch: in the product of any size, 1,011 rows x 6416 x 1760 took 217 us, 104 without.
template <bool SIDES = true>
__device__ __forceinline__ float both_sides(float x) {
  if constexpr (SIDES) asm volatile("" : "+v"(x));
  return x;
}
// exp(z) - 1 - z for z <= 0, the negative side of xIELU, without branches and no further from it than expm1f(z) - z: down to -1, where
// that difference cancels, z^2 times the polynomial that interpolates (exp(z) - 1 - z) / z^2 at seven Chebyshev nodes (9e-9
// relative with the coefficients in fp32); below, exp(z) - (1 + z) with exp(z) = 2^h (1 + l ln 2), h + l = z log2(e) to twice fp32's digits.  xIELU with it against
// 64 bits, root mean square of the relative error over z in [-1, 0] 1.1e-7 (1.5e-7 with expm1f), [-0.01, 0] 2.6e-8 (6.2e-8), [-100, -5]
// 1.1e-7 (the same).
template <bool SIDES = true>
__device__ __forceinline__ float expm1_less_z(float z) {
  const float p = z * z * (0.5f + z * (0.166666643f + z * (0.0416662902f + z * (0.00833105026f + z * (0.00138224157f + z * (0.000188324755f +
                  z * 1.69281272e-5f))))));
  const float t = fmaxf(z, -128.f);                          // (2^h is 0 long before; NaN stays in 1 + z)
  const float h = t * 1.44269502f, l = fmaf(t, 1.92596303e-8f, fmaf(t, 1.44269502f, -h));
  const float e = __builtin_amdgcn_exp2f(h);
  const float far = both_sides<SIDES>(fmaf(e, l * 0.693147182f, e) - (1.f + z));
  return z > -1.f ? both_sides<SIDES>(p) : far;
}
__device__ __forceinline__ float sigmoid_f(float z) { return 1.f / (1.f + expf(-z)); }
__device__ __forceinline__ float silu_f(float z) { return z / (1.f + expf(-z)); }
// gelu, tanh form: 0.5 z (1 + tanh(u)) with u = sqrt(2/pi) (z + 0.044715 z^3), written as z sigmoid(2u):
// one exponential, and no cancellation in the negative tail
__device__ __forceinline__ float gelu_tanh_f(float z) {
  return z / (1.f + expf(-1.5957691216057308f * (z + 0.044715f * z * z * z)));
}

// pooled blocks beside an attention window: one mean key and value for each block of P positions, rows of the block
// pools kp / vp (rows ldk / ldv wide, pages of the attention's page size, table[request][t_stride])
struct AttnBlocks {
  int P;
  const void* kp;
  int ldk;
  const void* vp;
  int ldv;
  const int* table;
  int t_stride;
};

// attn_paged.hip: out[t, h] from nsplit partial (maximum, sum, weighted values) records per (row, head)
typedef void* fls_stream_t;
// has_sink: the softmax's silent entry of score `sink` (sink_h given: sink_h[head]) joins the total here; head_gate (nullable) [T, H]: a sigmoid gate per (row, head)
int seq_attn_merge(const float* part, void* out, int tc, int ldo, int T, int H, int dv, int nsplit, int gated, float out_scale,
                   int has_sink, float sink, const float* sink_h, const float* head_gate, int ldhg, fls_stream_t s);

#define SEQ_LAUNCH_CHECK() do { hipError_t e_ = hipGetLastError(); if (e_ != hipSuccess) return (int)e_; } while (0)
