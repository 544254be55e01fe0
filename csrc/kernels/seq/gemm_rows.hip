// C[M,N] = epilogue(A[M,K] . W[N,K]^T) for few rows (decoding, small expert groups): a stream of W through the chip once.
//
// A block owns 16 output columns and its WV waves cut K between them, so that the loads of a whole column panel are in flight
// at once: a wave issues 16-byte loads of its 16 weight rows (and of the rows of A, which the caches hold) for eight K steps
// before the first of their MFMAs, straight from global memory -- nothing is read twice, LDS would only add a wait.  A K step
// is 32 elements of bf16 (one 16x16x32 MFMA) or 16 of fp32 (four 16x16x4 MFMAs, lane group g holding elements 4 g .. 4 g + 3).
// The waves' partial sums meet in LDS, in the order of the waves.  Bound by HBM: 8 rows against 32000 x 2048 bf16 take 32 us (4.1
// TB/s; 41 before), 2048 x 8192 16 us (43 before, four waves with two loads in flight each), in fp32 76 and 34 us (144 and 407
// on 64 x 64 tiles).
#include "seq_common.h"
#include "fls_seq.h"
#include "gemm_epi.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// what a lane holds of one K step: 8 bf16 or 4 fp32
template <typename TW> struct Step;
template <> struct Step<bf16_t> { typedef bf16x8 V; static constexpr int K = 32, LANE = 8; };
template <> struct Step<float> { typedef floatx4 V; static constexpr int K = 16, LANE = 4; };

__device__ __forceinline__ void load_step(const bf16_t* p, bf16x8& v) { v = *reinterpret_cast<const bf16x8*>(p); }
__device__ __forceinline__ void load_step(const float* p, floatx4& v) { v = *reinterpret_cast<const floatx4*>(p); }
__device__ __forceinline__ void load_step(const float* p, bf16x8& v) {        // fp32 rows against bf16 weights: rounded on the way in
  typedef float floatx8 __attribute__((ext_vector_type(8)));
  const floatx4 a = *reinterpret_cast<const floatx4*>(p), b = *reinterpret_cast<const floatx4*>(p + 4);
  const floatx8 f = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  v = __builtin_convertvector(f, bf16x8);
}
__device__ __forceinline__ floatx4 mfma_step(const bf16x8& w, const bf16x8& x, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, c, 0, 0, 0);
}
__device__ __forceinline__ floatx4 mfma_step(const floatx4& w, const floatx4& x, floatx4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], c, 0, 0, 0);
  return c;
}

template <typename TA, typename TW, int MG, int WV, bool GATED>
__global__ __launch_bounds__(64 * WV) void gemm_rows(const TA* __restrict__ A, const TW* __restrict__ W, void* __restrict__ C, Epi epi,
                                                     int M, int N, int K, int lda, int ldw, int ldc, const int* __restrict__ offs,
                                                     const int* __restrict__ a_rows, long long w_gs) {
  typedef typename Step<TW>::V V;
  constexpr int SK = Step<TW>::K, LN = Step<TW>::LANE, U = GATED ? 4 : 8, HW = GATED ? 2 : 1;
  __shared__ floatx4 red[WV][MG * HW][64];
  if (offs != nullptr) {                   // row groups (experts): this block's group owns rows offs[g] .. offs[g+1]
    const int g = blockIdx.y, r0 = offs[g];
    M = offs[g + 1] - r0;
    if (M <= 0) return;
    if (a_rows != nullptr) a_rows += r0;
    else A += (size_t)r0 * lda;
    C = reinterpret_cast<char*>(C) + (size_t)r0 * ldc * (epi.tc == 1 ? 2 : 4);
    W += (size_t)g * w_gs;
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15, grp = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int steps = (K + SK - 1) / SK, per = (steps + WV - 1) / WV;
  const int s0 = wave * per, s1 = min(steps, s0 + per);
  // (a gated product: the columns' gate rows and, N rows on, their up rows)
  const TW* wp[HW];
#pragma unroll
  for (int h = 0; h < HW; ++h) wp[h] = W + (size_t)(min(n0 + fr, N - 1) + h * N) * ldw + grp * LN;
  for (int m0 = 0; m0 < M; m0 += 16 * MG) {
    floatx4 acc[HW][MG];
    bool ok[MG];
    const TA* xp[MG];
#pragma unroll
    for (int u = 0; u < MG; ++u) {
#pragma unroll
      for (int h = 0; h < HW; ++h) acc[h][u] = floatx4{0.f, 0.f, 0.f, 0.f};
      const int r = min(m0 + u * 16 + fr, M - 1);
      ok[u] = m0 + u * 16 + fr < M;
      xp[u] = A + (size_t)(a_rows != nullptr ? a_rows[r] : r) * lda + grp * LN;
    }
    for (int s = s0; s < s1; s += U) {
      V w[HW][U], x[MG][U];
      bool in[U];                          // (the last step may end short: K is a multiple of a lane's share)
#pragma unroll
      for (int i = 0; i < U; ++i) {
        in[i] = s + i < s1 && (s + i) * SK + grp * LN < K;
#pragma unroll
        for (int h = 0; h < HW; ++h) {
          w[h][i] = V{};
          if (in[i]) load_step(wp[h] + (size_t)(s + i) * SK, w[h][i]);
        }
      }
#pragma unroll
      for (int u = 0; u < MG; ++u)
#pragma unroll
        for (int i = 0; i < U; ++i) {
          x[u][i] = V{};
          if (in[i] && ok[u]) load_step(xp[u] + (size_t)(s + i) * SK, x[u][i]);
        }
#pragma unroll
      for (int i = 0; i < U; ++i)
#pragma unroll
        for (int u = 0; u < MG; ++u)
#pragma unroll
          for (int h = 0; h < HW; ++h) acc[h][u] = mfma_step(w[h][i], x[u][i], acc[h][u]);
    }
    if (m0 > 0) __syncthreads();
#pragma unroll
    for (int u = 0; u < MG; ++u)
#pragma unroll
      for (int h = 0; h < HW; ++h) red[wave][u * HW + h][lane] = acc[h][u];
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * MG; i += 64 * WV) {
      const int u = i >> 6, l = i & 63;
      const int row = m0 + u * 16 + (l & 15), col0 = n0 + 4 * (l >> 4);
      if (row < M) {
        floatx4 v = red[0][u * HW][l], v2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 1; w < WV; ++w) v += red[w][u * HW][l];
        if constexpr (GATED) {
#pragma unroll
          for (int w = 0; w < WV; ++w) v2 += red[w][u * HW + 1][l];
        }
        EpiRegs er = epi_regs(epi);
        if constexpr (GATED) {
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const int col = col0 + x;
            if (col >= N) continue;
            const float o = epi_gate(v[x], v2[x], epi);
            if (epi.tc == 1) reinterpret_cast<bf16_t*>(C)[(size_t)row * ldc + col] = f_to_bf16(o);
            else reinterpret_cast<float*>(C)[(size_t)row * ldc + col] = o;
          }
        } else {
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const int col = col0 + x;
            if (col >= N) continue;
            epi_column(epi, er, col);
            v[x] = epi_value(v[x] + (epi.bias != nullptr ? epi.bias[col] : 0.f), epi, er);
            if (epi.tc == 1) reinterpret_cast<bf16_t*>(C)[(size_t)row * ldc + col] = f_to_bf16(v[x]);
            else reinterpret_cast<float*>(C)[(size_t)row * ldc + col] = v[x];
          }
          // (N is a multiple of 4 then: rows of N, 64 bytes of one a store)
          if (epi.mirror != nullptr && col0 < N) *reinterpret_cast<floatx4*>(*epi.mirror + (size_t)row * N + col0) = v;
        }
      }
    }
  }
}

template <typename TA, typename TW, int MG, int WV, bool GATED>
int start(const void* A, const void* W, void* C, const Epi& epi, int M, int N, int K, int lda, int ldw, int ldc, int groups, const int* offs,
          const int* a_rows, long long w_gs, hipStream_t s) {
  hipLaunchKernelGGL((gemm_rows<TA, TW, MG, WV, GATED>), dim3((N + 15) / 16, offs != nullptr ? groups : 1), dim3(64 * WV), 0, s, (const TA*)A,
                     (const TW*)W, C, epi, M, N, K, lda, ldw, ldc, offs, a_rows, w_gs);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 1 : -(int)e;
}

}  // namespace

int seq_gemm_rows(const void* A, int ta, const void* W, int tw, void* C, const Epi& epi, int M, int N, int K, int lda, int ldw, int ldc,
                  int groups, const int* offs, const int* a_rows, long long w_gs, hipStream_t s) {
  // Row groups of 16 rows a pass over W, or 32 (17 .. 32 rows in one pass: 24 x 2048 x 2048 8.1 us, 10.3 in two).  Eight waves share
  // K where one block a CU or less has all the columns (2048 columns: 6.4 us, 6.8 with four), four where several blocks share a CU
  // anyway (32000 columns: 32 us, 41 with eight; floor 28).
  const bool gated = epi.kind >= EPI_GATE;
  if (gated) N >>= 1;                      // columns of C
  const bool two = offs == nullptr && M > 16;
  const bool many = (long long)((N + 15) / 16) * (offs != nullptr ? groups : 1) > 256;
#define ROWS_AS(TA, TW, GATED)                                                                                            \
  (two ? (many ? start<TA, TW, 2, 4, GATED>(A, W, C, epi, M, N, K, lda, ldw, ldc, groups, offs, a_rows, w_gs, s)          \
               : start<TA, TW, 2, 8, GATED>(A, W, C, epi, M, N, K, lda, ldw, ldc, groups, offs, a_rows, w_gs, s))         \
       : (many ? start<TA, TW, 1, 4, GATED>(A, W, C, epi, M, N, K, lda, ldw, ldc, groups, offs, a_rows, w_gs, s)          \
               : start<TA, TW, 1, 8, GATED>(A, W, C, epi, M, N, K, lda, ldw, ldc, groups, offs, a_rows, w_gs, s)))
#define ROWS(TA, TW) (gated ? ROWS_AS(TA, TW, true) : ROWS_AS(TA, TW, false))
  if (tw == 0) return ROWS(float, float);
  return ta == 1 ? ROWS(bf16_t, bf16_t) : ROWS(float, bf16_t);
#undef ROWS
#undef ROWS_AS
}
