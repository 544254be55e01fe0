// What the matrix-product kernels (gemm_any.hip, gemm_tile.hip) do with a finished accumulator.
#pragma once
#include "seq_common.h"

// What a kernel does with a finished accumulator element: + bias, optionally an activation, then the store as fp32 or bf16 --
// so a projection whose consumer is the next matrix product writes that product's operand directly and the fp32
// intermediate never reaches memory.
//   1  xIELU with act = {p, q}: z > 0: softplus(p) z^2 + z/2, else (1/2 + softplus(q)) (exp(z) - 1 - z) + z/2
//   2  the square of max(z, 0)
//   3  a decay: exp(-exp(act[column / act_n]) softplus(z))
//   4  p tanh(z / p)
//   5  p z
//   6, 7, 8  a gated product: W holds [gate rows; up rows], N / 2 of each, C has N / 2 columns: silu(g) u, gelu(g) u (tanh
//      form), or g sigmoid(q g) (u + 1) with g = min(gate, p), u = clamp(up, -p, p)
enum { EPI_XIELU = 1, EPI_RELU2 = 2, EPI_DECAY = 3, EPI_SOFTCAP = 4, EPI_SCALE = 5, EPI_GATE = 6, EPI_LAST = 8 };
struct Epi {
  const float* bias;
  const float* act;      // the activation's numbers on the device, if it has any
  int kind;
  int tc;                // element type of C: 0 fp32, 1 bf16
  int act_n;             // kind 3: columns per number of act
  float p, q;
  float* const* mirror;  // where the fp32 results go as well (the cell, on the device, holds an address the device can write; null, here or there: nowhere)
};
struct EpiRegs { float ap, an; };
__device__ __forceinline__ EpiRegs epi_regs(const Epi& e) {
  EpiRegs r = {0.f, 0.f};
  if (e.kind == EPI_XIELU) { r.ap = softplus_f(e.act[0]); r.an = 0.5f + softplus_f(e.act[1]); }
  return r;
}
// (kind 3: what a lane's column needs, before its elements are emitted)
__device__ __forceinline__ void epi_column(const Epi& e, EpiRegs& r, int col) {
  if (e.kind == EPI_DECAY) r.ap = -expf(e.act[col / e.act_n]);
}
// exp(ap softplus(z)), ap <= 0, in units of log 2: softplus as max(z, 0) + log(1 + exp(-|z|)) in two terms, of which the hardware's exponential and logarithm
// give the first and exact residuals the second; near 1 a polynomial, where the exponential's last bit is the result's.  16 million
// behind an fp32 product of 64 terms 166 us by exp(ap log1p(exp(z))) and 104 so; from 64 bits, over normal z and ap of -1 .. -16, 3.3e-7 and 1.3e-7, largest 8.2e-6 and 1.3e-6.
// Infinities and numbers that no model has, whose terms leave the range of fp32, go by one product in their place.  mh and t are held as rounded: fused into
// the sums that follow, a product's rounding would be counted twice.  The code is short because kernels hold many copies of it: with the plain formula
// as a second path the kernel for any shape kept its accumulators in scratch.
__device__ __forceinline__ float decay_f(float ap, float z) {
  constexpr float L2E = 1.44269502f, L2E_LO = 1.92596299e-8f, LN2 = 0.693147181f;
  const float a = fmaxf(-fabsf(z), -130.f), h = a * L2E, hl = __builtin_fmaf(a, L2E, -h) + a * L2E_LO;
  const bool far = h < -125.f;             // (the hardware's exponential has no subnormal results)
  float e = __builtin_amdgcn_exp2f(far ? h + 64.f : h);
  e = __builtin_amdgcn_ldexpf(__builtin_fmaf(e, hl * LN2, e), far ? -64 : 0);
  const float u = 1.f + e, g = __builtin_amdgcn_logf(u), gl = (e - (u - 1.f)) * L2E * __builtin_amdgcn_rcpf(u);
  const float m = z < 0.f ? 0.f : z;       // (NaN stays)
  float mh = m * L2E;
  asm("" : "+v"(mh));
  const float ml = __builtin_fmaf(m, L2E, -mh) + m * L2E_LO, s = mh + g, sl = (g - (s - mh)) + (ml + gl);
  const bool out = z > 1e30f || ap < -1e30f;
  float t = ap * (out ? (z > 1e30f ? z : (s + sl) * LN2) : s);
  asm("" : "+v"(t));
  const float tl = out ? 0.f : t > -200.f ? __builtin_fmaf(ap, s, -t) + ap * sl : 0.f;
  if (out) t *= L2E;
  const bool low = t < -125.f;
  const float d = __builtin_amdgcn_exp2f(low ? t + 64.f : t), y = (t + tl) * LN2;
  const float near = __builtin_fmaf(y, __builtin_fmaf(y, __builtin_fmaf(y, __builtin_fmaf(y, 1.f / 24.f, 1.f / 6.f), 0.5f), 1.f), 1.f);
  return t > -0.0625f ? near : __builtin_amdgcn_ldexpf(__builtin_fmaf(d, tl * LN2, d), low ? -64 : 0);
}
template <int KIND, bool SIDES = true>
__device__ __forceinline__ float epi_value_of(float v, const Epi& e, const EpiRegs& r) {
  if constexpr (KIND == EPI_RELU2) { v = fmaxf(v, 0.f); return v * v; }
  else if constexpr (KIND == EPI_DECAY) return decay_f(r.ap, v);
  else if constexpr (KIND == EPI_XIELU) {
    const float low = both_sides<SIDES>(r.an * expm1_less_z<SIDES>(v));
    return (v > 0.f ? r.ap * v * v : low) + 0.5f * v;
  }
  else if constexpr (KIND == EPI_SOFTCAP) return e.p * tanhf(v / e.p);
  else if constexpr (KIND == EPI_SCALE) return v * e.p;
  else return v;
}
template <int KIND>
__device__ __forceinline__ float epi_gate_of(float g, float u, const Epi& e) {
  if constexpr (KIND == EPI_GATE) return silu_f(g) * u;
  else if constexpr (KIND == EPI_GATE + 1) return gelu_tanh_f(g) * u;
  g = fminf(g, e.p);
  u = fminf(fmaxf(u, -e.p), e.p);
  return g / (1.f + expf(-e.q * g)) * (u + 1.f);
}
__device__ __forceinline__ float epi_value(float v, const Epi& e, const EpiRegs& r) {
  if (e.kind == EPI_RELU2) return epi_value_of<EPI_RELU2>(v, e, r);
  if (e.kind == EPI_DECAY) return epi_value_of<EPI_DECAY>(v, e, r);
  if (e.kind == EPI_XIELU) return epi_value_of<EPI_XIELU, false>(v, e, r);
  if (e.kind == EPI_SOFTCAP) return epi_value_of<EPI_SOFTCAP>(v, e, r);
  if (e.kind == EPI_SCALE) return epi_value_of<EPI_SCALE>(v, e, r);
  return v;
}
__device__ __forceinline__ float epi_gate(float g, float u, const Epi& e) {
  if (e.kind == EPI_GATE) return epi_gate_of<EPI_GATE>(g, u, e);
  if (e.kind == EPI_GATE + 1) return epi_gate_of<EPI_GATE + 1>(g, u, e);
  return epi_gate_of<EPI_GATE + 2>(g, u, e);
}
__device__ __forceinline__ void emit(void* C, size_t idx, float v, const Epi& e) {
  if (e.tc == 1) reinterpret_cast<bf16_t*>(C)[idx] = f_to_bf16(v);
  else reinterpret_cast<float*>(C)[idx] = v;
}

// gemm_tile.hip: the product on LDS-DMA tiles; element types bf16 x bf16, fp32 x fp32, or fp32 rows against bf16 weights (rounded
// to them).  a_rows (nullable): row r of the product is made from row a_rows[r] of A.  Needs 16-byte-aligned rows of A and W.  1: launched; 0: not a shape it serves; < 0: failed.
int seq_gemm_tile(const void* A, int ta, const void* W, int tw, void* C, const Epi& epi, int M, int N, int K, int lda, int ldw, int ldc, int groups,
                  const int* offs, const int* a_rows, long long a_gs, int a_mod, long long w_gs, long long c_gs, hipStream_t s);

// gemm_rows.hip: the same for few rows.  Needs
// 16-byte-aligned rows of A and W.  1: launched; 0: not a shape it serves; < 0: failed.
int seq_gemm_rows(const void* A, int ta, const void* W, int tw, void* C, const Epi& epi, int M, int N, int K, int lda, int ldw, int ldc,
                  int groups, const int* offs, const int* a_rows, long long w_gs, hipStream_t s);
