// C[M,N] = epilogue(A[M,K] . W[N,K]^T) for few rows (decoding, small expert groups): a stream of W through the chip once.
//
// A block owns 16 output columns (or 32: NB = 2); its WV waves take the K tiles (128 bytes of a row) by turns, each with a ring of its own
// in LDS that DMAs fill, whole 128-byte lines of W's rows and of the rows of A that there are: no wave waits for another before the
// sums, which meet in LDS in the order of the waves.  A tile is two steps of 32 elements of bf16 (a 16x16x32 MFMA each) or 16 of fp32 (four
// 16x16x4 MFMAs, lane group g holding elements 4 g .. 4 g + 3).  Why not straight to registers: what a lane needs for an MFMA is 16 bytes of its own
// row, so that neighbouring lanes' loads are rows apart, and a CU takes such loads at 16 bytes a cycle, 54 by DMA; with the loads of A, as many for 16
// rows as for 16 columns, that was the bound.  Cold weights, before and so (us): 8 rows x 2048 x 2048 6.4, 5.2; x 2048 x 8192 15.1, 11.2; x 32000 x 2048
// 30.7, 26.8 (the rate of a copy: 27.8); 24 rows x 2048 x 2048 8.7, 6.2; x 2048 x 8192 23.3, 14.3; x 32000 x 2048 37.3, 30.1; gated 5440 x 2048 17.4, 12.9;
// fp32 8 rows x 2048 x 8192 27.8, 21.1, 24 rows 48.6, 30.3; 16 rows in 8 groups, gated 2048 x 2048 27.1, 24.3, 2048 x 2048 15.7, 14.2.
#include <algorithm>

#include "seq_common.h"
#include "fls_seq.h"
#include "gemm_epi.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// what a lane holds of one K step: 8 bf16 or 4 fp32
template <typename TW> struct Step;
template <> struct Step<bf16_t> { typedef bf16x8 V; };
template <> struct Step<float> { typedef floatx4 V; };

__device__ __forceinline__ floatx4 mfma_step(const bf16x8& w, const bf16x8& x, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, c, 0, 0, 0);
}
__device__ __forceinline__ floatx4 mfma_step(const floatx4& w, const floatx4& x, floatx4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], c, 0, 0, 0);
  return c;
}

#define LDS_AS __attribute__((address_space(3)))
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7fffffff, 0x00020000);
}
#define R_DMA(rs, off, k0, dst) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LDS_AS void*)(dst), 16, off, k0, 0, 0)

// A wave's ring: stages of a K tile of HW 16-row panels of W and of XR rows of A, 20 KB of them (eight waves on a CU, 64 KB of W and more in
// flight) for up to two rounds of blocks (one in fp32), else 10 KB and twice the blocks on a CU: 150 random products by row groups, many of them empty, took
// 0.93 (bf16), 0.87 (fp32 on bf16) and 0.86 (fp32) of their time before with 20 KB, 0.90, 0.85 and 0.82 with 10; 24 rows x 2048 x 8192 14.8 and 15.5 us,
// 48 rows of 10 groups x 2048 x 2048 20.0 and 20.6, 6 of 8 in fp32 21.3 and 20.0.
constexpr int stages_in(int bytes, int stage) { return bytes / stage < 2 ? 2 : bytes / stage > 6 ? 6 : bytes / stage; }
template <typename TA, typename TW, int XR, int HW> struct Ring {
  static constexpr int XS = sizeof(TA) / sizeof(TW), XA = XR * XS / 8, SW = HW * 2048, STAGE = SW + XA * 1024, CNT = 2 * HW + XA;
  static constexpr int NST = stages_in(20480, STAGE), FEW = stages_in(10240, STAGE);
};

// 16 bytes of a row, zeros where the offset is out of range
__device__ __forceinline__ floatx4 load16(__amdgpu_buffer_rsrc_t rs, unsigned off, int k0) {
  return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, k0, 0));
}
__device__ __forceinline__ bf16x8 rounded(const floatx4& lo, const floatx4& hi) {       // fp32 rows against bf16 weights
  typedef float floatx8 __attribute__((ext_vector_type(8)));
  return __builtin_convertvector((floatx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}), bf16x8);
}

// U > 0: operands straight to registers.  A short K is one chunk of U steps a wave, whose loads are all issued before the first product; what
// counts there is the chain of one load, and the way through LDS adds to it: 8 rows x 11808 x 224 4.0 us so, 4.4 by the rings.
template <typename TA, typename TW, int XR, int WV, int NB, bool GATED, int U>
__device__ __forceinline__ void rows_of(const TA* A, const TW* W, void* C, const Epi& epi, int M, int N, int K, int lda, int ldw, int ldc,
                                        const int* offs, const int* a_rows, long long w_gs, int nst) {
  typedef typename Step<TW>::V V;
  constexpr int HW = GATED ? 2 * NB : NB, MG = (XR + 15) / 16;
  typedef Ring<TA, TW, XR, HW> R;
  constexpr int XS = R::XS, XA = R::XA, STAGE = R::STAGE, NST = R::NST, CNT = R::CNT;
  extern __shared__ __attribute__((aligned(16))) char smem[];
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
  // DMA pieces of 1 KB: 8 rows of 128 bytes, 16-byte chunk c of row r in place c ^ (r & 7) (rows of A of twice the size: 4 rows, c ^ (r & 15))
  const int lr = lane >> 3, lc = (lane & 7) ^ lr;
  const int kb = K * (int)sizeof(TW), stages = (kb + 127) / 128, mine = (stages - wave + WV - 1) / WV;
  constexpr int SUMS = MG * HW * 1024;
  const int share = U > 0 ? SUMS : nst * STAGE;            // of LDS, a wave's
  char* const ring = smem + wave * share;
  __amdgpu_buffer_rsrc_t rw[HW];
  unsigned wo[HW][2];
#pragma unroll
  for (int h = 0; h < HW; ++h) {           // (a gated product: the columns' gate rows and, N rows on, their up rows)
    const int b = GATED ? h >> 1 : h, n1 = min(n0 + 16 * b, N - 1);
    const TW* p = W + (size_t)(n1 + (GATED && (h & 1) ? N : 0)) * ldw;
    rw[h] = rsrc_of(p);
#pragma unroll
    for (int j = 0; j < 2; ++j)
      wo[h][j] = (unsigned)min(U > 0 ? fr : 8 * j + lr, N - 1 - n1) * ldw * (unsigned)sizeof(TW) + (U > 0 ? grp : lc) * 16;
  }
  const __amdgpu_buffer_rsrc_t ra = rsrc_of(A);
  const bool few = XR == 16 && M <= 8;                     // (a row group: half of its stages' pieces of A)
  auto red = [&](int w, int at, int l) -> floatx4& { return *reinterpret_cast<floatx4*>(smem + w * share + (at * 64 + l) * 16); };
  static_assert(SUMS <= STAGE, "a wave's sums fit its ring");
  for (int m0 = 0; m0 < M; m0 += 16 * MG) {
    floatx4 acc[2][HW][MG];                // (the two steps of a tile in sums of their own, which rounds less)
#pragma unroll
    for (int u = 0; u < MG; ++u)
#pragma unroll
      for (int h = 0; h < HW; ++h) acc[0][h][u] = acc[1][h][u] = floatx4{0.f, 0.f, 0.f, 0.f};
    if constexpr (U > 0) {
      unsigned xo[MG];
#pragma unroll
      for (int u = 0; u < MG; ++u) {       // (rows past M: zeros, no loads)
        const int row = m0 + u * 16 + fr, r = min(row, M - 1);
        xo[u] = row < M ? (unsigned)(a_rows != nullptr ? a_rows[r] : r) * lda * (unsigned)sizeof(TA) + grp * (16 * XS) : 0x80000000u;
      }
      V w[HW][U], x[MG][U];
#pragma unroll
      for (int i = 0; i < U; ++i) {        // steps of 64 bytes of a row of W
        const int k0 = (wave * U + i) * 64;
        const unsigned none = k0 + grp * 16 >= kb ? 0x80000000u : 0u;
#pragma unroll
        for (int h = 0; h < HW; ++h) w[h][i] = __builtin_bit_cast(V, load16(rw[h], wo[h][0] | none, k0));
#pragma unroll
        for (int u = 0; u < MG; ++u) {
          const floatx4 lo = load16(ra, xo[u] | none, k0 * XS);
          if constexpr (XS == 1) x[u][i] = __builtin_bit_cast(V, lo);
          else x[u][i] = rounded(lo, load16(ra, (xo[u] + 16) | none, k0 * XS));
        }
      }
#pragma unroll
      for (int i = 0; i < U; ++i)
#pragma unroll
        for (int u = 0; u < MG; ++u)
#pragma unroll
          for (int h = 0; h < HW; ++h) acc[i & 1][h][u] = mfma_step(w[h][i], x[u][i], acc[i & 1][h][u]);
    } else {
      unsigned xo[XA];
#pragma unroll
      for (int i = 0; i < XA; ++i) {
        const int row = XS == 1 ? 8 * i + lr : 4 * i + (lane >> 4), r = min(m0 + row, M - 1);
        xo[i] = (unsigned)(a_rows != nullptr ? a_rows[r] : r) * lda * (unsigned)sizeof(TA) + (XS == 1 ? lc * 16 : ((lane ^ row) & 15) * 16);
      }
      auto fill = [&](int t, char* stg) {    // the wave's t-th stage (chunks past K: zeros)
        const int k0 = (wave + t * WV) * 128;
        const bool cut = k0 + 128 > kb;
        const unsigned none = cut && k0 + lc * 16 >= kb ? 0x80000000u : 0u;
#pragma unroll
        for (int h = 0; h < HW; ++h)
#pragma unroll
          for (int j = 0; j < 2; ++j) R_DMA(rw[h], wo[h][j] | none, k0, stg + (2 * h + j) * 1024);
#pragma unroll
        for (int i = 0; i < XA; ++i) {
          unsigned no = none;
          if (XS == 2) no = cut && k0 * 2 + (((lane ^ (4 * i + (lane >> 4))) & 15) * 16) >= kb * 2 ? 0x80000000u : 0u;
          if (!(few && i >= XA / 2)) R_DMA(ra, xo[i] | no, k0 * XS, stg + R::SW + i * 1024);
        }
      };
#pragma unroll
      for (int t = 0; t < NST; ++t)
        if (t < min(nst, mine)) fill(t, ring + t * STAGE);
      char* stg = ring;
      for (int t = 0; t < mine; ++t) {
        const int after = min(nst - 1, mine - 1 - t);        // stages that may stay in flight
        asm volatile("" ::: "memory");
#define R_VM(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | ((n) >> 4) << 14 | 0x0f70)
        if (after == 0) R_VM(0);
#define R_WAIT(n)                            \
    else if (NST > n && after == n) {          \
      if (few) R_VM(n * (CNT - XA / 2));       \
      else R_VM(n * CNT);                      \
    }
        R_WAIT(1)
        R_WAIT(2)
        R_WAIT(3)
        R_WAIT(4)
        R_WAIT(5)
#undef R_WAIT
#undef R_VM
        asm volatile("" ::: "memory");
        V w[HW][2], x[MG][2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int c = ((4 * k + grp) ^ (fr & 7)) << 4;
#pragma unroll
          for (int h = 0; h < HW; ++h) w[h][k] = *reinterpret_cast<const V*>(stg + h * 2048 + fr * 128 + c);
#pragma unroll
          for (int u = 0; u < MG; ++u) {
            const int r = min(u * 16 + fr, XR - 1);         // (rows past M: columns that are not stored)
            if constexpr (XS == 1) {
              x[u][k] = *reinterpret_cast<const V*>(stg + R::SW + r * 128 + (((4 * k + grp) ^ (r & 7)) << 4));
            } else {
              const char* row = stg + R::SW + r * 256;
              const int a = 8 * k + 2 * grp, sw = r & 15;
              const floatx4 lo = *(const floatx4*)(row + ((a ^ sw) << 4)), hi = *(const floatx4*)(row + (((a + 1) ^ sw) << 4));
              x[u][k] = rounded(lo, hi);
            }
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (t + nst < mine) fill(t + nst, stg);
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int u = 0; u < MG; ++u)
#pragma unroll
            for (int h = 0; h < HW; ++h) acc[k][h][u] = mfma_step(w[h][k], x[u][k], acc[k][h][u]);
        stg = stg + STAGE == ring + nst * STAGE ? ring : stg + STAGE;
      }
    }
#pragma unroll
    for (int u = 0; u < MG; ++u)
#pragma unroll
      for (int h = 0; h < HW; ++h) red(wave, u * HW + h, lane) = acc[0][h][u] + acc[1][h][u];
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * MG * NB; i += 64 * WV) {
      // (results that go to the host as well: neighbouring lanes write a row's columns, 64 NB bytes)
      const bool by_rows = host != nullptr;
      const int l = by_rows ? (i / (4 * NB) & 15) | (i & 3) << 4 : i & 63;
      const int b = by_rows ? (i >> 2) % NB : (i >> 6) % NB, u = (i >> 6) / NB, at = u * HW + (GATED ? 2 * b : b);
      const int row = m0 + u * 16 + (l & 15), col0 = n0 + 16 * b + 4 * (l >> 4);
      if (row < M) {
        floatx4 v = red(0, at, l), v2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 1; w < WV; ++w) v += red(w, at, l);
        if constexpr (GATED) {
#pragma unroll
          for (int w = 0; w < WV; ++w) v2 += red(w, at + 1, l);
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
          if (epi.bias != nullptr) {
#pragma unroll
            for (int x = 0; x < 4; ++x) v[x] += epi.bias[min(col0 + x, N - 1)];
          }
          // (one copy of the activations' code, out of plain products' way: a decode step runs some thirty kernels and finds none of them in the
          // instruction cache, so that plain products of 24 rows took 7.4 us there with four copies, 13 KB, and 6.7 with one, 7 KB)
          if (epi.kind != 0) {
#pragma unroll 1
            for (int x = 0; x < 4; ++x) {
              epi_column(epi, er, min(col0 + x, N - 1));
              v = floatx4{v[1], v[2], v[3], epi_value(v[0], epi, er)};
            }
          }
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const int col = col0 + x;
            if (col >= N) continue;
            if (epi.tc == 1) reinterpret_cast<bf16_t*>(C)[(size_t)row * ldc + col] = f_to_bf16(v[x]);
            else reinterpret_cast<float*>(C)[(size_t)row * ldc + col] = v[x];
          }
          // (N is a multiple of 4 then: rows of N, 64 bytes of one a store)
          if (host != nullptr && col0 < N) *reinterpret_cast<floatx4*>(host + (size_t)row * N + col0) = v;
        }
      }
    }
    if (m0 + 16 * MG < M) __syncthreads();               // (the sums lie in the rings)
  }
}

template <typename TA, typename TW, int XR, int WV, int NB, bool GATED, int U>
__global__ __launch_bounds__(64 * WV) void gemm_rows(const TA* __restrict__ A, const TW* __restrict__ W, void* __restrict__ C, Epi epi,
                                                     int M, int N, int K, int lda, int ldw, int ldc, const int* __restrict__ offs,
                                                     const int* __restrict__ a_rows, long long w_gs, int nst) {
  rows_of<TA, TW, XR, WV, NB, GATED, U>(A, W, C, epi, M, N, K, lda, ldw, ldc, offs, a_rows, w_gs, nst);
}

template <typename TA, typename TW, int XR, int WV, int NB, bool GATED, int U>
int start(const void* A, const void* W, void* C, const Epi& epi, int M, int N, int K, int lda, int ldw, int ldc, int groups, const int* offs,
          const int* a_rows, long long w_gs, hipStream_t s) {
  typedef Ring<TA, TW, XR, GATED ? 2 * NB : NB> R;
  constexpr int SUMS = (XR + 15) / 16 * (GATED ? 2 * NB : NB) * 1024;
  static const hipError_t a = hipFuncSetAttribute((const void*)gemm_rows<TA, TW, XR, WV, NB, GATED, U>, hipFuncAttributeMaxDynamicSharedMemorySize, WV * (U > 0 ? SUMS : R::NST * R::STAGE));
  if (a != hipSuccess) return -(int)a;
  const int cols = (N + 16 * NB - 1) / (16 * NB), gs = offs != nullptr ? groups : 1, stages = (K * (int)sizeof(TW) + 127) / 128;
  const bool deep = (long long)cols * gs <= (sizeof(TW) == 2 ? 1024 : 512);
  int nst = std::min((int)(deep ? R::NST : R::FEW), (stages + WV - 1) / WV);       // (a short K needs less)
  const int fit = 163840 / (WV * 2 * R::STAGE);            // blocks of two large stages a wave that a CU's LDS holds: where there are more, one stage and twice the blocks
  if (nst == 2 && fit <= 2 && (stages <= 2 * WV || (fit == 1 && !GATED)) && (long long)cols * std::min(gs, M) > 256 * fit) nst = 1;
  hipLaunchKernelGGL((gemm_rows<TA, TW, XR, WV, NB, GATED, U>), dim3(cols, gs), dim3(64 * WV), WV * (U > 0 ? SUMS : nst * R::STAGE), s, (const TA*)A, (const TW*)W,
                     C, epi, M, N, K, lda, ldw, ldc, offs, a_rows, w_gs, nst);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 1 : -(int)e;
}

}  // namespace

int seq_gemm_rows(const void* A, int ta, const void* W, int tw, void* C, const Epi& epi, int M, int N, int K, int lda, int ldw, int ldc,
                  int groups, const int* offs, const int* a_rows, long long w_gs, hipStream_t s) {
  // 16 rows a pass over W (8 if there are no more in all), without row groups up to 32 in one.  Eight waves share K where one block a CU or less
  // has all the columns and K is more than a tile for each (8 rows x 2048 x 2048 5.2 us, 5.3 with four; 24 rows 6.2 and 6.2, gated 7.2 and 7.0),
  // else four, two blocks a CU or more.  Blocks of 32 columns read half as much of A and leave no half-empty second round: from one round of
  // 16-column blocks (below it 1.04 to 1.4 of the time) to 448 (8 rows x 6416 x 2048 8.3 -> 7.8 us; of 1,500 random widths of 200 to 720 blocks 0.9 to 0.95 of the
  // time up to 320, 0.83 to 1.05 to 448, and from 480 to 512 on slower but for the next kinds), plain products of more than 16 rows above that too (24 rows x
  // 8192 x 2048 10.2 -> 9.5, x 32000 32.8 -> 30.1; fp32 from 512 to 720 blocks is 1.1 to 1.19 so), plain ones of more than 8 fp32 rows on bf16 weights above 1024
  // blocks (16,400 to 66,000 columns 0.90 to 0.94; bf16 rows 0.96 to 1.03, up to 8 rows 0.97 to 1.08), and plain row groups of a row each or more on bf16
  // weights (48 rows of 10 x 2048 x 2048 19.9 -> 18.9; 4 rows of 8 8.0 and 7.7).
  const bool gated = epi.kind >= EPI_GATE;
  if (gated) N >>= 1;                      // columns of C
  const int ea = ta == 1 ? 2 : 4, ew = tw == 1 ? 2 : 4;
  if (((long long)ldw * 16 + 8) * ew >= (1LL << 31) || (long long)lda * M * ea >= (1LL << 31)) return 0;      // (32-bit offsets within a panel, among the rows)
  const bool two = offs == nullptr && M > 16;
  const long long blocks = (long long)((N + 15) / 16) * (offs != nullptr ? groups : 1);
  const bool wide = offs != nullptr ? !gated && tw == 1 && M >= groups : blocks > 256 && (blocks <= 448 || (!gated && (two || (ta != tw && M > 8 && blocks > 1024))));
  const bool eight = !two && !gated && blocks <= 256 && K * ew > 512;
  // Straight to registers, in one chunk of 1, 2 or 3 steps for each of four waves (10,000 random products, times by the rings' with their spread over classes of rows
  // and blocks): up to 256 bytes of a row of W 0.78 - 0.97, to 512 0.90 - 0.99 without gated row groups (1.00 - 1.04), to 768 0.92 - 1.02 for plain
  // products of up to 16 rows and row groups; with eight waves to 1024 for those of up to 16 rows in a round of blocks (0.93 - 0.96).  A block reads its
  // rows of A beside 16 columns: where that is more than 32 KB a CU in all, the rings' wider blocks are as fast or faster (1.1 - 1.4 above 1,500 blocks).
  const int kb = K * ew;
  const bool light = offs != nullptr || blocks <= 256 || blocks * ((gated ? 32 : 16) * kb + (long long)M * K * ea) <= 256 * 32768;
  const int steps = !light ? 0 : kb <= 256 ? 1 : kb <= 512 && !(gated && offs != nullptr) ? 2 : kb <= 768 && !gated && !two ? 3 : 0;
  const bool direct = steps > 0 || (kb <= 1024 && offs == nullptr && eight);
#define START(TA, TW, XR, WV, NB, GATED, U) start<TA, TW, XR, WV, NB, GATED, U>(A, W, C, epi, M, N, K, lda, ldw, ldc, groups, offs, a_rows, w_gs, s)
#define PANELS(TA, TW, XR)                                                                                                 \
  (gated ? (wide ? START(TA, TW, XR, 4, 2, true, 0) : START(TA, TW, XR, 4, 1, true, 0))                                    \
         : wide ? START(TA, TW, XR, 4, 2, false, 0) : eight ? START(TA, TW, XR <= 16 ? XR : 16, 8, 1, false, 0) : START(TA, TW, XR, 4, 1, false, 0))
#define CHUNK(TA, TW, U)                                                                                                   \
  (two ? (gated ? START(TA, TW, 32, 4, 1, true, U) : START(TA, TW, 32, 4, 1, false, U))                                    \
       : gated ? START(TA, TW, 16, 4, 1, true, U) : START(TA, TW, 16, 4, 1, false, U))
#define CHUNKS(TA, TW)                                                                                                     \
  (steps == 1 ? CHUNK(TA, TW, 1) : steps == 2 ? CHUNK(TA, TW, 2) : steps == 3 ? START(TA, TW, 16, 4, 1, false, 3) : START(TA, TW, 16, 8, 1, false, 2))
#define ROWS(TA, TW)                                                                                                       \
  (direct ? CHUNKS(TA, TW) : two ? (M <= 24 ? PANELS(TA, TW, 24) : PANELS(TA, TW, 32)) : M <= 8 ? PANELS(TA, TW, 8) : PANELS(TA, TW, 16))
  if (tw == 0) return ROWS(float, float);
  return ta == 1 ? ROWS(bf16_t, bf16_t) : ROWS(float, bf16_t);
#undef ROWS
#undef CHUNKS
#undef CHUNK
#undef PANELS
#undef START
}
