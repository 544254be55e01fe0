// C[M,N] = epilogue(A[M,K] . W[N,K]^T) for few rows (decoding, small expert groups): a stream of W through the chip once.
//
// A block owns 16 output columns (or 32: NB = 2) and its WV waves cut K between them in chunks of U steps: a wave issues a chunk's
// 16-byte loads of its weight rows, and of the rows of A that there are (the caches hold them), before the first of their MFMAs, straight
// from global memory -- nothing of W is read twice, LDS would only add a wait.  A K step is 32 elements of bf16 (one 16x16x32 MFMA) or 16
// of fp32 (four 16x16x4 MFMAs, lane group g holding elements 4 g .. 4 g + 3).  The waves' partial sums meet in LDS, in the order of the waves.
// What bounds it is HBM where the weight is large, else the chain of a launch, a load's latency and the sums (2048 x 2048: 6.3 us); what
// keeps the loads in flight is many waves with few registers each, not long chunks: with two or four steps a chunk (row groups: twice), no masks on whole chunks
// and 32-bit offsets a wave takes 58 to 116 registers (blocks of 32 columns 130 to 148; eight steps: 98 to 156).  Cold weights, eight steps and here: 8 rows x 8192 x 2048
// 12.6 -> 10.0 us, 6416 x 2048 13.5 -> 9.9, 32000 x 2048 32 -> 30.7 (floor 28); 24 rows x 6416 x 2048 14.7 -> 12.1, gated 5440 x 2048 20.2 -> 18.1;
// fp32, 3 rows x 2048 x 8192 29.9 -> 27.3, 32000 x 2048 59.6 -> 51.4.  A second chunk's registers, loaded ahead, were slower everywhere.  What is
// left of K behind the whole chunks is one chunk with masks (step by step, each waiting for its loads: 21 rows x 6416 x 736 8.7 us, 7.1 so).
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

template <typename TA, typename TW, int MG, int WV, int U, int NB, bool GATED>
__global__ __launch_bounds__(64 * WV) void gemm_rows(const TA* __restrict__ A, const TW* __restrict__ W, void* __restrict__ C, Epi epi,
                                                     int M, int N, int K, int lda, int ldw, int ldc, const int* __restrict__ offs,
                                                     const int* __restrict__ a_rows, long long w_gs) {
  typedef typename Step<TW>::V V;
  constexpr int SK = Step<TW>::K, LN = Step<TW>::LANE, HW = GATED ? 2 * NB : NB;
  __shared__ floatx4 red[WV][MG * HW][64];
  float* const host = !GATED && epi.mirror != nullptr ? *epi.mirror : nullptr;
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
  const int n0 = blockIdx.x * 16 * NB;
  const int steps = (K + SK - 1) / SK, chunks = (steps + U - 1) / U, per = (chunks + WV - 1) / WV * U;
  const int s0 = wave * per, s1 = min(steps, s0 + per);
  // (a gated product: the columns' gate rows and, N rows on, their up rows)
  const TW* wb[HW];
  unsigned wo[HW];
#pragma unroll
  for (int h = 0; h < HW; ++h) {
    const int b = GATED ? h >> 1 : h, n1 = min(n0 + 16 * b, N - 1);
    wb[h] = W + (size_t)(n1 + (GATED && (h & 1) ? N : 0)) * ldw;
    wo[h] = (unsigned)(min(fr, N - 1 - n1) * ldw + grp * LN);
  }
  for (int m0 = 0; m0 < M; m0 += 16 * MG) {
    floatx4 acc[HW][MG];
    bool ok[MG];
    const TA* xp[MG];
    V x[MG][U];
#pragma unroll
    for (int u = 0; u < MG; ++u) {
#pragma unroll
      for (int h = 0; h < HW; ++h) acc[h][u] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < U; ++i) x[u][i] = V{};             // (rows past M stay zero: no loads for them)
      const int r = min(m0 + u * 16 + fr, M - 1);
      ok[u] = m0 + u * 16 + fr < M;
      xp[u] = A + (size_t)(a_rows != nullptr ? a_rows[r] : r) * lda + grp * LN;
    }
    int s = s0;
    for (; s + U <= s1 && (s + U) * SK <= K; s += U) {
      V w[HW][U];
#pragma unroll
      for (int i = 0; i < U; ++i)
#pragma unroll
        for (int h = 0; h < HW; ++h) load_step(wb[h] + s * SK + (wo[h] + i * SK), w[h][i]);
#pragma unroll
      for (int u = 0; u < MG; ++u)
        if (ok[u]) {
#pragma unroll
          for (int i = 0; i < U; ++i) load_step(xp[u] + (size_t)(s + i) * SK, x[u][i]);
        }
#pragma unroll
      for (int i = 0; i < U; ++i)
#pragma unroll
        for (int u = 0; u < MG; ++u)
#pragma unroll
          for (int h = 0; h < HW; ++h) acc[h][u] = mfma_step(w[h][i], x[u][i], acc[h][u]);
    }
    if (s < s1) {                          // (the last chunk may end short, and its last step: K is a multiple of a lane's share)
      V w[HW][U];
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const bool in = s + i < s1 && (s + i) * SK + grp * LN < K;
#pragma unroll
        for (int h = 0; h < HW; ++h) {
          w[h][i] = V{};
          if (in) load_step(wb[h] + s * SK + (wo[h] + i * SK), w[h][i]);
        }
#pragma unroll
        for (int u = 0; u < MG; ++u) {
          x[u][i] = V{};
          if (in && ok[u]) load_step(xp[u] + (size_t)(s + i) * SK, x[u][i]);
        }
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
    for (int i = threadIdx.x; i < 64 * MG * NB; i += 64 * WV) {
      // (results that go to the host as well: neighbouring lanes write a row's columns, 64 NB bytes)
      const bool by_rows = host != nullptr;
      const int l = by_rows ? (i / (4 * NB) & 15) | (i & 3) << 4 : i & 63;
      const int b = by_rows ? (i >> 2) % NB : (i >> 6) % NB, u = (i >> 6) / NB, at = u * HW + (GATED ? 2 * b : b);
      const int row = m0 + u * 16 + (l & 15), col0 = n0 + 16 * b + 4 * (l >> 4);
      if (row < M) {
        floatx4 v = red[0][at][l], v2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 1; w < WV; ++w) v += red[w][at][l];
        if constexpr (GATED) {
#pragma unroll
          for (int w = 0; w < WV; ++w) v2 += red[w][at + 1][l];
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
          if (host != nullptr && col0 < N) *reinterpret_cast<floatx4*>(host + (size_t)row * N + col0) = v;
        }
      }
    }
  }
}


template <typename TA, typename TW, int MG, int WV, int U, int NB, bool GATED>
int start(const void* A, const void* W, void* C, const Epi& epi, int M, int N, int K, int lda, int ldw, int ldc, int groups, const int* offs,
          const int* a_rows, long long w_gs, hipStream_t s) {
  hipLaunchKernelGGL((gemm_rows<TA, TW, MG, WV, U, NB, GATED>), dim3((N + 16 * NB - 1) / (16 * NB), offs != nullptr ? groups : 1), dim3(64 * WV), 0, s,
                     (const TA*)A, (const TW*)W, C, epi, M, N, K, lda, ldw, ldc, offs, a_rows, w_gs);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 1 : -(int)e;
}

}  // namespace

int seq_gemm_rows(const void* A, int ta, const void* W, int tw, void* C, const Epi& epi, int M, int N, int K, int lda, int ldw, int ldc,
                  int groups, const int* offs, const int* a_rows, long long w_gs, hipStream_t s) {
  // Row groups of 16 rows a pass over W, or 32 (17 .. 32 rows in one pass: 24 x 2048 x 2048 8.1 us, 10.3 in two).  Eight waves share
  // K where one block a CU or less has all the columns (2048 x 8192: 15.4 us, 17.2 with four), four where several blocks share a CU
  // anyway (8192 x 2048: 10.0, 10.8 with eight).  With two row groups a block of 16 columns reads twice as much of A as of W: 32 from 6,400
  // columns on (24 rows x 6416 x 2048: 14.1 us -> 12.1, x 32000 44.7 -> 37.9; 4096 x 14336 38.6, 50 on 128 blocks).  9,700 random products
  // (profiles/cases/few_rows_columns.txt): 1.2 to 1.3 of the time up to 4,096 columns, 0.8 to 0.96 from there to 8,176, 0.9 to 1.15 above.
  // Row groups: most of a launch's blocks may belong to empty groups, and the others have their CU to themselves: twice the steps in flight (of
  // 10,200 random products 0.7% are more than 6% slower than on eight steps, gated four; with the short chunks 12%, up to 1.5 times).
  const bool gated = epi.kind >= EPI_GATE;
  if (gated) N >>= 1;                      // columns of C
  if ((long long)ldw * 16 + 8 >= (1LL << 31)) return 0;      // (32-bit offsets within a panel)
  const bool two = offs == nullptr && M > 16;
  const bool many = (long long)((N + 15) / 16) * (offs != nullptr ? groups : 1) > 256;
#define START(TA, TW, MG, WV, U, NB, GATED) start<TA, TW, MG, WV, U, NB, GATED>(A, W, C, epi, M, N, K, lda, ldw, ldc, groups, offs, a_rows, w_gs, s)
#define ROWS(TA, TW)                                                                                                       \
  (gated ? (two ? (many ? START(TA, TW, 2, 4, 2, 1, true) : START(TA, TW, 2, 8, 2, 1, true))                               \
                : (many ? (offs != nullptr ? START(TA, TW, 1, 4, 4, 1, true) : START(TA, TW, 1, 4, 2, 1, true))            \
                        : START(TA, TW, 1, 8, 4, 1, true)))                                                                \
         : (two ? (N >= 6400 ? START(TA, TW, 2, 4, 4, 2, false)                                                            \
                             : many ? START(TA, TW, 2, 4, 4, 1, false) : START(TA, TW, 2, 8, 4, 1, false))                 \
                : (many ? (offs != nullptr ? START(TA, TW, 1, 4, 8, 1, false) : START(TA, TW, 1, 4, 4, 1, false))          \
                        : START(TA, TW, 1, 8, 4, 1, false))))
  if (tw == 0) return ROWS(float, float);
  return ta == 1 ? ROWS(bf16_t, bf16_t) : ROWS(float, bf16_t);
#undef ROWS
#undef START
}
