// MFMA GEMM for the Llama projections on gfx950 (MI355X / CDNA4).
//
//   C[M, N'] = epilogue( A[M, K] . W[N, K]^T )      fp16 in, fp32 accumulate
//
// A = activations (tokens x hidden, row-major), W = nn.Linear weight [out, in]
// (row-major, exactly as stored in the checkpoint) — both operands are
// K-contiguous, the natural MFMA layout.  The weights are consumed in the
// checkpoint's own row order: nothing is permuted on the host or by a relayout
// pass, so a layer streams from disk to HBM as plain DMA (runtime/stream.py).
//
// Kernels (one C ABI entry, fls_gemm, picks by shape):
//   * gemm_nt_v10 — 256 x 256 x 64 tile, 4 waves (one per SIMD), each wave
//     128 x 128 outputs in 256 AGPR accumulators (v_mfma_f32_16x16x32_f16: holds
//     a higher clock than 32x32x16 on random data, guide §5.4 r28).  Operands
//     staged global -> LDS by buffer_load_dwordx4 ... lds (LDS-DMA) with the XOR
//     chunk swizzle on the per-lane SOURCE address (guide T2 / rule 21), three
//     half-tile super-phases in flight, one counted vmcnt + raw s_barrier per
//     two phases, LDS fragment reads and DMA interleaved into the MFMA stream.
//     XCD-aware bijective block remap + grouped tile order (guide T1).
//   * gemm_nt_col16 — blocks of 16 columns or pairs of columns, for M <= 64 and narrow outputs;
//   * gemm_nt_mid — 64 x 128 x 64 tiles, 3-deep LDS-DMA ring, for M too small
//     to fill 256 CUs with 256 x 256 tiles, and for odd K-tile counts (v10's
//     body is unrolled over two K-tiles); 4 waves, or 8 (two per SIMD) for
//     grids of about one block per CU, 64 or 128 rows; 64-column blocks.
//   * gemm_nt_generic — any shape (bounds-masked loads), for odd test shapes.
//
// The MFMA computes C^T tiles (A operand = W fragment, B operand = X fragment)
// so each lane holds 4 consecutive output columns of one row in each 16-column
// subtile (v10 pairs neighbouring subtiles into 16-byte stores with one
// v_permlane16_swap), and the epilogue partners live in the same lane:
//   RESID : C = acc (+ bias) + R          (R may alias C: in-place residual)
//   SWIGLU: W = [gate (I rows); up (I rows)] (HF gate_proj / up_proj stacked);
//           the W-tile loader reads logical rows interleaved per 16 (gate rows
//           16j.., up rows 16j..) so gate and up of one intermediate column sit
//           in neighbouring subtiles of the same lane; C has I = N/2 columns,
//           silu(gate) * up.
//   ROPE  : HF rotate-half on every head of the first rope_cols columns, in
//           natural head-dim order: the partner of column d of a head is
//           d + head_dim/2, which is 4 (hd 128) or 2 (hd 64) subtiles further
//           in the same lane; fp32 cos/sin tables [maxpos, hd/2], pos[m].
#include "gemm_v10.h"

extern "C" int fls_gemm_v11_pays(int M, int N);      // gemm_v11.hip

namespace {

// ------------------------------------------------------------- generic
// Block = 4 waves; block tile 32 (M) x 256 (N); wave tile 32 x 64.
// Operands loaded straight from global with bounds masks (zero fill).
template <int EPI>
__global__ __launch_bounds__(256) void gemm_nt_generic(const half_t* __restrict__ A, const half_t* __restrict__ W,
                                                     half_t* __restrict__ C, int M, int N, int K, int lda, int ldw,
                                                     int ldc, Epi ep) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int fr = lane & 15, grp = lane >> 4;
  const int m0 = blockIdx.x * 32;
  const bool rope128 = EPI == FLS_EPI_ROPE;
  // 128-column group of this wave and its position in it
  const int gbase = blockIdx.y * 256 + (wave >> 1) * 128;
  int ncol[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) ncol[t] = gbase + sub_col(rope128, wave & 1, t);
  floatx4 acc[2][4];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[u][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += 32) {
    half8 wf[4], xf[2];
    const int kb = k0 + grp * 8;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int n = ncol[t] + fr;
      const int nr = EPI == FLS_EPI_SWIGLU ? gu_phys_row(n, ep.gu_rows) : n;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        wf[t][j] = (n < N && kb + j < K) ? W[(size_t)nr * ldw + kb + j] : (half_t)0.f;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int m = m0 + u * 16 + fr;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        xf[u][j] = (m < M && kb + j < K) ? A[(size_t)m * lda + kb + j] : (half_t)0.f;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[u][t] = mfma16x16x32(wf[t], xf[u], acc[u][t]);
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int m = m0 + u * 16 + fr;
    if (m >= M) continue;
    if constexpr (is_rope(EPI)) {
#pragma unroll
      for (int q = 0; q < 2; ++q)
        if (ncol[q + 2] + 16 <= N) store_rope_pair(C, ldc, m, ncol[q] + 4 * grp, acc[u][q], acc[u][q + 2], ep);
    } else {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int nf = ncol[2 * p];
        if (nf + 32 <= N) {
          store_pair_off<EPI>(C, ldc, m, nf, 4 * grp, acc[u][2 * p], acc[u][2 * p + 1], ep);
        } else if constexpr (EPI == FLS_EPI_NONE || EPI == FLS_EPI_RESID) {
          // ragged tail (N % 32 != 0): scalar stores
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int n = nf + h * 16 + 4 * grp + r;
              if (n < N) {
                float v = (h ? acc[u][2 * p + 1][r] : acc[u][2 * p][r]) * row_scale(ep, m);
                if (ep.bias) v += (float)ep.bias[n];
                if constexpr (EPI == FLS_EPI_RESID) v = v * ep.alpha + (float)ep.R[(size_t)m * ep.ldr + n];
                C[(size_t)m * ldc + n] = (half_t)v;
              }
            }
        }
      }
    }
  }
}

// ------------------------------------------------------------------ mid-M
// For small / medium M (a few prompts, generation steps, LM heads with > 16
// scored rows) the 256x256 tiles leave most of the 256 CUs idle (7B QKV at
// M = 416: 96 blocks).  gemm_nt_mid uses 64 (M) x 128 (N) x 64 tiles: 4 waves
// in a 2 x 2 grid, each 32 x 64 outputs (2 x 4 MFMA 16x16x32 tiles, 32 fp32
// accumulators), operands staged by LDS-DMA (16 B per lane, XOR chunk swizzle
// on the source address) into a 3-deep ring with one counted vmcnt + raw
// barrier per K-tile; XCD-aware order puts every M tile of one N tile on the
// same XCD so each weight tile comes from HBM once and from L2 after that.
// Any K-tile count (the tail path for odd K / 64).
// One 16-column subtile of row m (columns c0 .. c0+3 of this lane): store_pair_off's arithmetic for
// one of its two subtiles, so 32-column mid blocks give the same bits (NONE / RESID epilogues)
template <int EPI>
__device__ __forceinline__ void store_one(half_t* __restrict__ C, int ldc, int m, int c0, const floatx4& acc,
                                          const Epi& ep) {
  static_assert(EPI == FLS_EPI_NONE || EPI == FLS_EPI_RESID, "pair epilogues need both subtiles");
  const float s = row_scale(ep, m);
  floatx4 a = acc * s;
  if (ep.bias) {
    const half4 ba = *(const half4*)(ep.bias + c0);
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] += (float)ba[r];
  }
  if constexpr (EPI == FLS_EPI_RESID) {
    const half4 ra = *(const half4*)(ep.R + (size_t)m * ep.ldr + c0);
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = a[r] * ep.alpha + (float)ra[r];
  }
  half4 oa;
#pragma unroll
  for (int r = 0; r < 4; ++r) oa[r] = (half_t)a[r];
  *(half4*)(C + (size_t)m * ldc + c0) = oa;
}

// 8-wave 64-row mid blocks: column (in the 128-column block) of subtile t of wave column wn.  RoPE: the
// pair is a column and its partner hd/2 away (hd 128: 64 columns; hd 64: 32 in the same head).
__device__ __forceinline__ int mid8_col(int epi, int wn, int t) {
  if (epi == FLS_EPI_ROPE) return wn * 16 + t * 64;
  if (epi == EPI_ROPE64) return (wn >> 1) * 64 + (wn & 1) * 16 + t * 32;
  return wn * 32 + t * 16;
}

namespace mid {
constexpr int BMm = 64, BNm = 128, BKm = 64, NTm = 256, NSTAGE = 3;
// BNT: output columns per block, 128 (4 waves in 2 x 2, each 32 x 64) or 64 (each 32 x 32: twice the
// blocks for grids of less than one round of 128-column tiles); 32 with 8 waves (below)
// A rows 0 .. bmt-1 then W rows; LDS-DMA in groups of 1 KiB: 8 rows, of K-tiles of 128 terms 4
constexpr int stage_bytes(int bnt, int bmt = BMm, int bk = BKm) { return (bmt + bnt) * bk * 2; }
}  // namespace mid

// NST: LDS stages, NST - 1 K-tiles in flight ahead of the one being multiplied (3: 72 KB, two blocks
// per CU).  A 6-stage ring for one-round grids measured the same (70B generation-step shapes at
// M = 16-320, profiles/r6_decode/mid_ring): the blocks are not bound by their DMA latency.
// BNT = 64 blocks: a wave holds two 16-column subtiles (RoPE: a column and its partner hd/2 away; for
// head_dim 128 a block takes 32 columns of a head and their 32 partners).  Same fragments, MFMA and
// K order as BNT = 128, so the two are bitwise equal.
//
// WV = 8, two waves per SIMD.  With grids of about one block per CU (generation steps: the O / down /
// QKV projections at M = 16-320) a 4-wave block is bound by the latency chain of its single wave per
// SIMD (DMA wait, barrier, LDS reads, MFMAs); a second wave's MFMAs run under the first one's LDS
// reads (70B down at M = 160: 225 -> 196 us).  Shapes:
//   BMT = 64 : waves in 2 x 4, each 32 x 32 outputs (its two 16-column subtiles are a RoPE pair: a
//              column and its partner hd/2 away); 72 KB of LDS, two blocks per CU;
//   BMT = 128: waves in 4 x 2, each 32 x 64 as in the 4-wave block; 96 KB, one block per CU, half the
//              blocks (M = 320: 192 instead of 320, which left 64 CUs with two blocks);
//   BNT = 64 : waves in 4 x 2, each 16 x 32 (the 4-wave 64-column block's columns); M <= 64 layers
//              406 -> 377 us at M = 16, 431 -> 417 at M = 64 (profiles/r6_decode/mid8/bn64_*);
//   BNT = 32 : waves in 4 x 2, each 16 x 16 (plain / residual epilogues): 70B down at M = 64
//              155 -> 139 us (profiles/r6_decode/mid8/bn32_*).
// Same fragments, MFMA and K order in every shape, so all are bitwise equal.
//
// BNT = 64 and 128, WV = 8: K-tiles of BK = 128 (64 where K is no multiple of it), one barrier a K-tile: after it tile kt - 1 has been
// read, so that its stage takes the tile NST - 1 ahead.  What bounds these grids of one row tile is the chain of one K-tile in few blocks
// a CU: M = 24, 50 and 64 (us, with K-tiles of 64 and two barriers, and so) 12,288 x 4,096 27.9, 29.2, 28.2 -> 24.3, 27.1, 26.0; 10,240 x
// 8,192 49.2, 51.1, 52.1 -> 42.8, 46.9, 49.4 with three stages (one block a CU); 22,016 x 4,096 43.4, 47.5, 49.6 -> 43.2, 46.3, 48.2 with
// two stages (two blocks; 47.6, 49.5, 51.0 with three). So BNT = 128 up to a round of blocks and from 2,048 terms on (1,024: 1.03 of the
// time): M = 65, 128 x 12,288 x 4,096 30.7, 35.2 -> 28.9, 33.3; 150, 256 x 4,096 x 11,008 71.6, 79.0 -> 66.8, 72.8; 192 x 8,192 x 4,096
// 31.1 -> 29.8.
template <int EPI, int NST, int BNT, int WV = 4, int BMT = mid::BMm, int BK = 64>
__global__ __launch_bounds__(64 * WV) void gemm_nt_mid(const half_t* __restrict__ A, const half_t* __restrict__ W,
                                                     half_t* __restrict__ C, int M, int N, int K, int lda, int ldw,
                                                     int ldc, Epi ep) {
  using namespace mid;
  static_assert(WV == 4 || WV == 8, "4 or 8 waves");
  static_assert(BNT != 32 || (WV == 8 && (EPI == FLS_EPI_NONE || EPI == FLS_EPI_RESID)),
                "32-column blocks: 8 waves, one 16-column subtile per wave (no pair epilogues)");
  static_assert(BMT == 64 || (BMT == 128 && WV == 8 && BNT == 128), "128-row blocks: 8 waves, 128 columns");
  constexpr bool L24 = WV == 8 && BMT == 64 && BNT == 128;   // 2 x 4 waves of 32 x 32
  constexpr bool L42 = WV == 8 && BNT <= 64;                 // 4 x 2 waves of 16 x 32 (x 16 at BNT 32)
  constexpr int RW = L42 ? 16 : 32, U = RW / 16;             // rows per wave, 16-row subtiles per wave
  constexpr bool ONE = WV == 8 && (BNT == 64 || BK == 128);  // one barrier a K-tile
  constexpr int LPR = BK / 8, RPD = 64 / LPR, KM = LPR - 1;  // lanes (16-byte chunks) a row, rows a DMA group of 1 KB
  // LDS-DMA groups: waves 0 .. NG % WV - 1 take one more when they do not divide evenly
  constexpr int NG = (BMT + BNT) / RPD, PER_WAVE = (NG + WV - 1) / WV, NG_REM = NG % WV;
  static_assert(!ONE || NG_REM == 0, "one count of DMAs");
  constexpr int STAGE = stage_bytes(BNT, BMT, BK), NSUB = L24 ? 2 : BNT == 32 ? 1 : BNT / 32;
  extern __shared__ __attribute__((aligned(16))) char lds_mid[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15, grp = lane >> 4;
  const int mt = (M + BMT - 1) / BMT, ntn = N / BNT;
  // XCD-aware bijective remap: logical tiles [xcd*q .. ) run on one XCD, M fastest
  int bid = blockIdx.x;
  {
    const int nwg = mt * ntn;
    const int q = nwg >> 3, r = nwg & 7, xcd = bid & 7, loc = bid >> 3;
    if (nwg >= 8) bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + loc;
  }
  const int m0 = (bid % mt) * BMT;
  const int bn = bid / mt;
  const int n0 = bn * BNT;
  const int wm = L24 ? wave >> 2 : wave >> 1, wn = L24 ? wave & 3 : wave & 1;
  const int nk = K / BK;
  const bool rope128 = EPI == FLS_EPI_ROPE;
  // BNT = 64 with RoPE over 128-wide heads: local W row l -> column of head bn / 2, quarter bn % 2
  const bool split_head = BNT == 64 && rope128;
  auto gcol = [&](int l) -> int {
    if (split_head) return (bn >> 1) * 128 + (bn & 1) * 32 + (l < 32 ? l : 64 + (l - 32));
    return n0 + l;
  };

  // this lane's LDS-DMA sources: group g = wave + WV*i covers tile rows RPD*g .. RPD*g+RPD-1
  const half_t* src[PER_WAVE];
  const int sub = lane / LPR;                      // row inside the group
#pragma unroll
  for (int i = 0; i < PER_WAVE; ++i) {
    const int g = min(wave + WV * i, NG - 1);       // (a group past NG is never issued)
    const int kc = ((lane ^ (g * RPD + sub)) & KM) * 8;           // source chunk pre-swizzled (read XORs it back)
    if (g < BMT / RPD) {
      const int m = min(m0 + g * RPD + sub, M - 1);
      src[i] = A + (size_t)m * lda + kc;
    } else {
      const int n = gcol((g - BMT / RPD) * RPD + sub);
      const int nr = EPI == FLS_EPI_SWIGLU ? gu_phys_row(n, ep.gu_rows) : n;
      src[i] = W + (size_t)nr * ldw + kc;
    }
  }
  // stage s takes K-tile kt (kt clamped to the last: a DMA past the end re-reads it into a stage
  // nobody reads again, so every wait is one constant count)
  auto stage = [&](int s, int kt) {
    char* base = lds_mid + (s % NST) * STAGE;
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i)
      if (NG_REM == 0 || i < PER_WAVE - 1 || wave < NG_REM)   // wave-uniform
        glds16(src[i] + (size_t)kt * BK, base + (wave + WV * i) * 1024);
  };
  // local W rows of this wave's subtiles (RoPE: subtile t + NSUB / 2 is subtile t's partner)
  int wrow[NSUB];
#pragma unroll
  for (int t = 0; t < NSUB; ++t) {
    if constexpr (L24) wrow[t] = mid8_col(EPI, wn, t) + fr;
    else if constexpr (BNT == 128) wrow[t] = sub_col(rope128, wn, t) + fr;
    else if constexpr (BNT == 32) wrow[t] = wn * 16 + fr;
    else wrow[t] = (is_rope(EPI) ? wn * 16 + t * 32 : wn * 32 + t * 16) + fr;
  }

  floatx4 acc[U][NSUB];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int t = 0; t < NSUB; ++t) acc[u][t] = floatx4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int d = 0; d < NST - 1; ++d) stage(d, min(d, nk - 1));
  for (int kt = 0; kt < nk; ++kt) {
    if constexpr (ONE) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * PER_WAVE) : "memory");
      __builtin_amdgcn_s_barrier();                        // every wave's part of tile kt landed; tile kt - 1 has been read
      asm volatile("" ::: "memory");
    }
    // into the stage tile kt - 1 used (every wave passed the barrier behind its reads: the one above, or that tile's closing one)
    stage(kt + NST - 1, min(kt + NST - 1, nk - 1));
    // tile kt landed
    if constexpr (!ONE) {
      if (NG_REM == 0 || wave < NG_REM) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 1) * PER_WAVE) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 1) * (PER_WAVE - 1)) : "memory");
      __builtin_amdgcn_s_barrier();                        // every wave's part of tile kt landed
    }
    const char* Xs = lds_mid + (kt % NST) * STAGE;
    const char* Ws = Xs + BMT * BK * 2;
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      const int c = ks * 4 + grp;                          // logical 16-byte chunk of this lane
      half8 xf[U], wf[NSUB];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r = wm * RW + u * 16 + fr;
        xf[u] = *(const half8*)(Xs + r * (BK * 2) + ((c ^ (r & KM)) << 4));
      }
#pragma unroll
      for (int t = 0; t < NSUB; ++t) {
        const int r = wrow[t];
        wf[t] = *(const half8*)(Ws + r * (BK * 2) + ((c ^ (r & KM)) << 4));
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < NSUB; ++t) acc[u][t] = mfma16x16x32(wf[t], xf[u], acc[u][t]);
    }
    // WAR: the next iteration's DMA overwrites this stage; all reads are done
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if constexpr (!ONE) __builtin_amdgcn_s_barrier();
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // the redundant tail DMA, before LDS is handed on
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int m = m0 + wm * RW + u * 16 + fr;
    if (m >= M) continue;
    if constexpr (L24) {
      if constexpr (is_rope(EPI))
        store_rope_pair(C, ldc, m, n0 + mid8_col(EPI, wn, 0) + 4 * grp, acc[u][0], acc[u][1], ep);
      else
        store_pair_off<EPI>(C, ldc, m, n0 + wn * 32, 4 * grp, acc[u][0], acc[u][1], ep);
    } else if constexpr (BNT == 32) {
      store_one<EPI>(C, ldc, m, n0 + wn * 16 + 4 * grp, acc[u][0], ep);
    } else if constexpr (is_rope(EPI)) {
      if constexpr (BNT == 128) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
          store_rope_pair(C, ldc, m, n0 + sub_col(rope128, wn, q) + 4 * grp, acc[u][q], acc[u][q + 2], ep);
      } else {
        store_rope_pair(C, ldc, m, gcol(wn * 16) + 4 * grp, acc[u][0], acc[u][1], ep);
      }
    } else {
#pragma unroll
      for (int p = 0; p < NSUB / 2; ++p)
        store_pair_off<EPI>(C, ldc, m, n0 + wn * (BNT / 2) + p * 32, 4 * grp, acc[u][2 * p], acc[u][2 * p + 1], ep);
    }
  }
}

// Blocks of 16 columns (the O / down projections of a 7B-sized generation step, N = 4,096: 128 mid blocks of 32 columns), or of two panels
// of 16 (neighbours, or pairs: a RoPE column and its partner, a gate and its up column), for M <= 64.  What bounds the wider mid blocks there is the
// bytes in flight: one block's ring on half of the CUs, with 64 rows of A staged whatever M is.
// Here a block streams 16 or 32 weight rows in K-tiles of 256 or 128 (two or four rows a DMA instruction, XOR chunk swizzle on the source) through
// a ring of NST stages with one barrier a K-tile; of two panels a CU has two blocks.  Only ceil(M / 16) row tiles of A are staged, wave w multiplies
// row tile w, the others only move data.  Same fragments, MFMA and K order as the mid blocks: bitwise equal rows.
// One panel, M = 16, K = 4,096 and 11,008 in turn (124 MB in both): 35.8 -> 16.6 us on average, 13 at the rate of a large copy.
// Pairs (us, 64-column mid blocks and these), M = 16: 22,016 x 4,096 42.5, 35.2; 12,288 x 4,096 26.1, 25.3; 6,144 x 4,096 22.5, 14.9;
// 5,120 x 2,048 12.7, 7.6; M = 64, the last two: 23.9, 19.7 and 13.8, 11.4.
// Two panels, plain, 16 rows (32-column mid blocks before): 8,192 x 8,192 45.1, 33.1; 8,192 x 28,672 147, 88.
// (A ring for W and a shorter one for A, loaded by waves of their own: 1.5 to 2 us slower.)
namespace col16 {
constexpr int kt(int rt, int np) { return np == 2 && rt > 1 ? 128 : 256; }
constexpr int stage_bytes(int rt, int np) { return 16 * (np + rt) * kt(rt, np) * 2; }
constexpr int stages(int rt, int np) { return np == 2 ? (rt == 2 ? 5 : 3) : rt == 1 ? 8 : rt == 2 ? 6 : 3; }       // 128 / 144 / 120 KB; pairs 72 / 80 / 72
}  // namespace col16

//
// STAT (up to 32 rows): the row statistic that the epilogue applies is made here, from the rows of A that pass through LDS anyway, by the
// waves that only move data (a wave for each part of 128 columns of a K-tile), in row_stat_kernel's order (same bits): a lane has one
// row's column group, its parts stay in registers, four to a lane group, and are added as warp_sum adds them.  A launch less for every
// norm + projection of a generation step.  us with that launch in front and so: 16 rows x 12,288 x 4,096 27.8, 26.0; x 22,016 x 4,096
// 36.9, 35.1; x 10,240 x 8,192 44.8, 42.9; x 6,144 x 2,048 10.4, 8.6; 32 rows x 6,144 x 2,048 11.3, 10.4.  (Both parts of a tile in one
// wave: x 22,016 36.6.  Above 32 rows the multiplying waves would have to make it: 48 rows 12.8, 15.1.)
template <int EPI, int RT, int NP, bool STAT>
__global__ __launch_bounds__(256) void gemm_nt_col16(const half_t* __restrict__ A, const half_t* __restrict__ W,
                                                   half_t* __restrict__ C, int M, int N, int K, int lda, int ldw,
                                                   int ldc, Epi ep) {
  constexpr int KT = col16::kt(RT, NP), NST = col16::stages(RT, NP), STAGE = col16::stage_bytes(RT, NP);
  constexpr int LPR = KT / 8, RPD = 64 / LPR, GP = 16 / RPD;               // lanes a row, rows a DMA group of 1 KB, groups a panel of 16 rows
  constexpr int PER_WAVE = GP * (NP + RT) / 4;           // DMA groups of a stage, per wave
  extern __shared__ __attribute__((aligned(16))) char lds_c16[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15, grp = lane >> 4;
  const int b = blockIdx.x, nk = K / KT;
  // a pair's second column is hd / 2 rows on (SwiGLU: I rows; no pairs: the next 16)
  const int n0 = EPI == FLS_EPI_ROPE ? (b >> 2) * 128 + (b & 3) * 16 : EPI == EPI_ROPE64 ? (b >> 1) * 64 + (b & 1) * 16
                 : b * (EPI == FLS_EPI_SWIGLU ? 16 : 16 * NP);
  const int second = EPI == FLS_EPI_ROPE ? 64 : EPI == EPI_ROPE64 ? 32 : EPI == FLS_EPI_SWIGLU ? ep.gu_rows : 16;
  const half_t* src[PER_WAVE];                         // groups 0 .. GP NP - 1: W rows, panel by panel, then A rows
#pragma unroll
  for (int i = 0; i < PER_WAVE; ++i) {
    const int g = wave + 4 * i, row = g % GP * RPD + lane / LPR;           // row inside its panel
    const int kc = ((lane % LPR) ^ row) * 8;
    src[i] = g < GP * NP ? W + (size_t)(n0 + (NP == 2 && g >= GP ? second : 0) + row) * ldw + kc
                         : A + (size_t)min((g / GP - NP) * 16 + row, M - 1) * lda + kc;
  }
  auto stage = [&](int s, int kt) {
    char* base = lds_c16 + (s % NST) * STAGE;
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) glds16(src[i] + (size_t)kt * KT, base + (wave + 4 * i) * 1024);
  };
  floatx4 acc[NP];
#pragma unroll
  for (int h = 0; h < NP; ++h) acc[h] = floatx4{0.f, 0.f, 0.f, 0.f};
  constexpr int SPW = KT / 128;                          // parts of 128 columns in a K-tile: a wave each
  static_assert(!STAT || RT * (1 + SPW) <= 4, "waves beside those that multiply");
  const int srt = (wave - RT) / SPW, spart = (wave - RT) % SPW;             // row tile and part whose statistics the wave makes
  const bool stat = STAT && wave >= RT && srt < RT;
  const int srow = ((NP + srt) * 16 + fr) * KT * 2;
  unsigned so[8];                                        // a part's columns 32 p + 4 grp + 16 h of the row: 16-byte chunk 4 p + 2 h + grp / 2, half of it
#pragma unroll
  for (int x = 0; x < 8; ++x) so[x] = (((2 * x + (grp >> 1)) ^ fr) << 4) + (grp & 1) * 8;
  float sp[STAT ? 16 : 1];
#pragma unroll
  for (int r = 0; r < (STAT ? 16 : 1); ++r) sp[r] = 0.f;
#pragma unroll
  for (int d = 0; d < NST - 1; ++d) stage(d, min(d, nk - 1));
  for (int kt = 0; kt < nk; ++kt) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * PER_WAVE) : "memory");
    __builtin_amdgcn_s_barrier();                      // every wave's part of tile kt landed; tile kt - 1 has been read
    asm volatile("" ::: "memory");
    stage(kt + NST - 1, min(kt + NST - 1, nk - 1));    // (past the end: the last tile again, into a stage nobody reads)
    if (wave < RT) {
      const char* Ws = lds_c16 + (kt % NST) * STAGE + fr * (KT * 2);
      const char* Xs = Ws + (NP + wave) * 16 * KT * 2;
      half8 wf[NP][KT / 32], xf[KT / 32];
#pragma unroll
      for (int ks = 0; ks < KT / 32; ++ks) {
        const int c = ((ks * 4 + grp) ^ fr) << 4;
#pragma unroll
        for (int h = 0; h < NP; ++h) wf[h][ks] = *(const half8*)(Ws + h * (16 * KT * 2) + c);
        xf[ks] = *(const half8*)(Xs + c);
      }
#pragma unroll
      for (int ks = 0; ks < KT / 32; ++ks)
#pragma unroll
        for (int h = 0; h < NP; ++h) acc[h] = mfma16x16x32(wf[h][ks], xf[ks], acc[h]);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if (stat) {
      const unsigned xs = (unsigned)(size_t)(__attribute__((address_space(3))) char*)lds_c16 + (kt % NST) * STAGE + srow + spart * 256;
      half4 q[8];                                        // (in asm: of loads of its own the compiler believes that they want every DMA landed)
      asm volatile("ds_read_b64 %0, %8\n\tds_read_b64 %1, %9\n\tds_read_b64 %2, %10\n\tds_read_b64 %3, %11\n\t"
                   "ds_read_b64 %4, %12\n\tds_read_b64 %5, %13\n\tds_read_b64 %6, %14\n\tds_read_b64 %7, %15\n\ts_waitcnt lgkmcnt(0)"
                   : "=&v"(q[0]), "=&v"(q[1]), "=&v"(q[2]), "=&v"(q[3]), "=&v"(q[4]), "=&v"(q[5]), "=&v"(q[6]), "=&v"(q[7])
                   : "v"(xs + so[0]), "v"(xs + so[1]), "v"(xs + so[2]), "v"(xs + so[3]), "v"(xs + so[4]), "v"(xs + so[5]), "v"(xs + so[6]), "v"(xs + so[7])
                   : "memory");
      float sq = 0.f;
#pragma unroll
      for (int p = 0; p < 4; ++p) sq = ss_accum_pair(sq, q[2 * p], q[2 * p + 1]);
      sq = row_sum_4groups(sq);
      const int part = kt * SPW + spart;                 // lane group part % 4, register part / 4
      if ((part & 3) == grp) {
#pragma unroll
        for (int r = 0; r < (STAT ? 16 : 1); ++r) sp[r] = (part >> 2) == r ? sq : sp[r];
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const int m = wave * 16 + fr;
  // (of ep itself but for the statistic: of a copy the compiler loads what it needs from the arguments only here, a trip to memory after
  // another: residual products of up to 3,000 columns 0.3 us slower)
  auto finish = [&](const Epi& e) {
    if (wave >= RT || m >= M) return;
    if constexpr (NP == 1) store_one<EPI>(C, ldc, m, n0 + 4 * grp, acc[0], e);
    else if constexpr (is_rope(EPI)) store_rope_pair<true>(C, ldc, m, n0 + 4 * grp, acc[0], acc[1], e);
    else store_pair_off<EPI>(C, ldc, m, b * 32, 4 * grp, acc[0], acc[1], e);
  };
  if constexpr (STAT) {
    __syncthreads();                                     // (every wave's DMAs have landed and its reads are done)
    float* const sums = reinterpret_cast<float*>(lds_c16) + 64;
    if (stat) {
#pragma unroll
      for (int o = 8; o > 0; o >>= 1)
#pragma unroll
        for (int r = 0; r < o; ++r) sp[r] += sp[r + o];
      if (SPW == 2 && (grp & 1) == spart) sums[srt * 64 + lane] = sp[0];          // (a wave's parts lie in every other lane group)
    }
    if constexpr (SPW == 2) __syncthreads();
    if (stat && spart == 0) {
      const float v = row_sum_4groups(SPW == 2 ? sums[srt * 64 + lane] : sp[0]);
      if (grp == 0) reinterpret_cast<float*>(lds_c16)[srt * 16 + fr] = rsqrtf(v / (float)K + ep.rs_eps);
    }
    __syncthreads();
    Epi e2 = ep;
    e2.rs = reinterpret_cast<const float*>(lds_c16);
    finish(e2);
  } else {
    finish(ep);
  }
}

template <int EPI, int RT, int NP, bool STAT = false>
void launch_col16(const half_t* A, const half_t* W, half_t* C, int M, int N, int K, int lda, int ldw, int ldc,
                  const Epi& ep, hipStream_t s) {
  constexpr int lds = col16::stages(RT, NP) * col16::stage_bytes(RT, NP);
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)gemm_nt_col16<EPI, RT, NP, STAT>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    attr = true;
  }
  hipLaunchKernelGGL((gemm_nt_col16<EPI, RT, NP, STAT>), dim3(N / (16 * NP)), dim3(256), lds, s, A, W, C, M, N, K, lda, ldw, ldc, ep);
}

int g_order = 0;             // 0: by shape, else a fixed signed group size (fls_gemm_set_order)
int g_mid = 1;               // mid-M kernel on (fls_gemm_set_mid)
int g_mid_bn = 0;            // mid-M block columns: 0 auto, 64 / 128 forced where valid (fls_gemm_set_mid_bn)
int g_mid_waves = 0;         // 128-column mid blocks: 0 auto, 4 / 8 waves forced (fls_gemm_set_mid_waves)
int g_mid_rows = 0;          // 8-wave mid blocks' rows: 0 auto, 64 / 128 forced (fls_gemm_set_mid_rows)

template <int EPI, int NST, int BNT, int WV = 4, int BMT = mid::BMm, int BK = 64>
void launch_mid(const half_t* A, const half_t* W, half_t* C, int M, int N, int K, int lda, int ldw, int ldc,
                const Epi& ep, hipStream_t s) {
  static bool attr = false;
  constexpr int lds = NST * mid::stage_bytes(BNT, BMT, BK);
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)gemm_nt_mid<EPI, NST, BNT, WV, BMT, BK>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    attr = true;
  }
  const int blocks = ((M + BMT - 1) / BMT) * (N / BNT);
  hipLaunchKernelGGL((gemm_nt_mid<EPI, NST, BNT, WV, BMT, BK>), dim3(blocks), dim3(64 * WV), lds, s, A, W, C, M, N, K,
                     lda, ldw, ldc, ep);
}

template <int EPI, int HX>
void launch_rows(const half_t* A, const half_t* W, half_t* C, int M, int N, int K, int lda, int ldw, int ldc, Epi ep,
                 hipStream_t s) {
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)gemm_nt_v10<EPI, false, HX>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              2 * v10_stage(HX));
    attr = true;
  }
  const int tiles_m = (M + 64 * HX - 1) / (64 * HX), tiles_n = N / BN;
  ep.order = g_order ? g_order : auto_order(tiles_m, tiles_n);
  hipLaunchKernelGGL((gemm_nt_v10<EPI, false, HX>), dim3(tiles_m * tiles_n), dim3(256), 2 * v10_stage(HX), s, A, W, C,
                     M, N, K, lda, ldw, ldc, ep);
}

int g_v10_rows = 0;          // rows of a v10 tile: 0 by shape (v10_rows), 128, 192 or 256 forced (fls_gemm_set_v10_rows)

template <int EPI>
void launch_main(int rows, const half_t* A, const half_t* W, half_t* C, int M, int N, int K, int lda, int ldw,
                 int ldc, const Epi& ep, hipStream_t s) {
  if (rows == 128) launch_rows<EPI, 2>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
  else if (rows == 192) launch_rows<EPI, 3>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
  else launch_rows<EPI, 4>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
}


// ------------------------------------------------------------ split-K
// Small M (generation steps, small calls): a 256 x 256 tile grid of a few dozen tiles leaves most
// CUs idle and the mid-M kernel's 64-row tiles re-read every weight panel once per row tile.  Here
// each tile's K is cut into S slices (tiles x S >= one block per CU), every block streams its slice
// of the weight panel ONCE (the activation slice comes from L2) and writes fp32 partials
// (gemm_nt_v10<EPI_F32>); splitk_reduce_kernel sums the S slabs in a fixed order (deterministic)
// and applies the real epilogue (bias, residual, SwiGLU on the natural [gate; up] columns, RoPE
// with the partner column d + hd/2 of each head).
constexpr int SPLITK_MAX_M = 512;
int g_splitk = 1;            // split-K path for small M on (fls_gemm_set_splitk)
int ROW_CHUNK = 16384;       // main-path launches cover at most this many rows (fls_gemm_set_row_chunk)

template <int EPI>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int S, long long pstride,
                                                            int M, int N, half_t* __restrict__ C, int ldc, Epi ep) {
  const int units = N / 4;                                   // 4 raw columns per thread
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long long)M * units) return;
  const int m = (int)(idx / units), c = (int)(idx % units) * 4;
  const float rsc = row_scale(ep, m);
  auto sum4 = [&](int col) {
    floatx4 a = *(const floatx4*)(part + (size_t)m * N + col);
    for (int k = 1; k < S; ++k) a += *(const floatx4*)(part + (size_t)k * pstride + (size_t)m * N + col);
    return a * rsc;
  };
  auto bias4 = [&](floatx4& a, int col) {
    if (ep.bias) {
      const half4 b = *(const half4*)(ep.bias + col);
#pragma unroll
      for (int r = 0; r < 4; ++r) a[r] += (float)b[r];
    }
  };
  auto store4 = [&](const floatx4& a, int col) {
    half4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = (half_t)a[r];
    *(half4*)(C + (size_t)m * ldc + col) = o;
  };
  if constexpr (EPI == FLS_EPI_SWIGLU) {
    const int I = N / 2;
    if (c >= I) return;                                      // gate threads do both halves
    const floatx4 g = sum4(c), u = sum4(I + c);
    floatx4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = silu(g[r]) * u[r];
    store4(o, c);
  } else if constexpr (is_rope(EPI)) {
    const int hd = ep.head_dim, half_hd = hd >> 1, d = c % hd;
    if (c < ep.rope_cols && d >= half_hd) return;            // the partner thread rotates this pair
    floatx4 a = sum4(c);
    bias4(a, c);
    if (c >= ep.rope_cols) {
      store4(a, c);
      return;
    }
    floatx4 b = sum4(c + half_hd);
    bias4(b, c + half_hd);
    const int p = ep.pos[m];
    const floatx4 cs = *(const floatx4*)(ep.cos_t + (size_t)p * half_hd + d);
    const floatx4 sn = *(const floatx4*)(ep.sin_t + (size_t)p * half_hd + d);
    floatx4 y1, y2;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      y1[r] = a[r] * cs[r] - b[r] * sn[r];
      y2[r] = b[r] * cs[r] + a[r] * sn[r];
    }
    store4(y1, c);
    store4(y2, c + half_hd);
  } else {
    floatx4 a = sum4(c);
    bias4(a, c);
    if constexpr (EPI == FLS_EPI_RESID) {
      const half4 rr = *(const half4*)(ep.R + (size_t)m * ep.ldr + c);
#pragma unroll
      for (int r = 0; r < 4; ++r) a[r] = a[r] * ep.alpha + (float)rr[r];
    }
    store4(a, c);
  }
}

#include "gemm_skinny.h"

// ss[m * ss_ld + j] = sum over columns [128 j, 128 j + 128) of C[m, :]^2 (fp32 of the fp16 values):
// the per-row partials of the v10 / v11 residual epilogue (Epi::ss) for the GEMM paths whose own
// epilogue does not write them (skinny, split-K, mid-M, generic: small M), and the fused norm's
// statistic of a hidden state without partials (fls_row_ss).  One wave per (16 rows, 128 columns) in
// the epilogue's lane layout -- lane (row fr, group g) holds columns 32 p + 4 g + r and 32 p + 16 +
// 4 g + r, p, r < 4 -- through the same ss_accum_pair and row_sum_4groups: bitwise the epilogue's.
__global__ __launch_bounds__(256) void ss_partials_kernel(const half_t* __restrict__ C, int ldc, int M, int nparts,
                                                          float* __restrict__ ss, int ss_ld) {
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int rgroups = (M + 15) / 16;
  if (w >= rgroups * nparts) return;                // wave-uniform
  const int fr = lane & 15, grp = lane >> 4;
  const int m = (w / nparts) * 16 + fr, j = w % nparts;
  const half_t* p0 = C + (size_t)min(m, M - 1) * ldc + j * 128 + grp * 4;
  float sq = 0.f;
#pragma unroll
  for (int p = 0; p < 4; ++p) sq = ss_accum_pair(sq, *(const half4*)(p0 + p * 32), *(const half4*)(p0 + p * 32 + 16));
  sq = row_sum_4groups(sq);                         // every lane (permlane swaps)
  if (grp == 0 && m < M) ss[(size_t)m * ss_ld + j] = sq;
}

// the fused norm's statistic straight from x: the 128-column parts of a row with ss_partials_kernel's per-lane FMA chains (one per
// 4-column group g) combined as row_sum_4groups does, (g0 + g2) + (g1 + g3), and summed in rstd_from_ss_kernel's order
// (lane j takes parts j, j + 64, ..., then warp_sum): the same bits as fls_row_ss followed by fls_rstd_from_ss, in one launch.
// What bounds it is one row's chain: four lanes a part, one for each of its column groups, 128 lanes a row (us, a lane for a whole part
// before: 65 rows of 4,096 3.03 -> 2.58, of 8,192 3.68 -> 2.90, 6,400 of 4,096 14.8 -> 10.7; one row 2.06 -> 2.21).
constexpr int ROW_STAT_MAX_PARTS = 128;              // H <= 16,384
__global__ __launch_bounds__(256) void row_stat_kernel(const half_t* __restrict__ x, int ldx, int M, int nparts, int H,
                                                       float eps, float* __restrict__ rstd) {
  __shared__ float parts[2][ROW_STAT_MAX_PARTS];
  const int r = threadIdx.x >> 7, l = threadIdx.x & 127, g = l & 3, m = blockIdx.x * 2 + r;
  const half_t* row = x + (size_t)min(m, M - 1) * ldx + 4 * g;
  for (int j = l >> 2; j < nparts; j += 32) {
    half4 q[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) q[k] = *(const half4*)(row + j * 128 + k * 16);
    float sq = 0.f;
#pragma unroll
    for (int p = 0; p < 4; ++p) sq = ss_accum_pair(sq, q[2 * p], q[2 * p + 1]);
    sq += __shfl_xor(sq, 2, 64);
    sq += __shfl_xor(sq, 1, 64);                    // (g0 + g2) + (g1 + g3)
    if (g == 0) parts[r][j] = sq;
  }
  __syncthreads();
  if (l >= 64 || m >= M) return;                    // wave-uniform
  float v = 0.f;
  for (int j = l; j < nparts; j += 64) v += parts[r][j];
  v = warp_sum(v);
  if (l == 0) rstd[m] = rsqrtf(v / (float)H + eps);
}

void row_stat(const half_t* x, int ldx, int rows, int H, float eps, float* rstd, hipStream_t s) {
  hipLaunchKernelGGL(row_stat_kernel, dim3((rows + 1) / 2), dim3(256), 0, s, x, ldx, rows, H / 128, H, eps, rstd);
}

void ss_partials_raw(const half_t* C, int ldc, int M, int N, float* ss, int ss_ld, hipStream_t s) {
  if (!ss || M <= 0) return;
  const int waves = ((M + 15) / 16) * (N / 128);
  hipLaunchKernelGGL(ss_partials_kernel, dim3((waves + 3) / 4), dim3(256), 0, s, C, ldc, M, N / 128, ss, ss_ld);
}

void ss_partials(const half_t* C, int ldc, int M, int N, const Epi& ep, hipStream_t s) {
  ss_partials_raw(C, ldc, M, N, ep.ss, ep.ss_ld, s);
}

// -> slices per tile (0: split-K not applicable / no room in the workspace)
int splitk_slices(int M, int N, int K, size_t tiles, size_t ws_bytes) {
  if (tiles >= 128) return 0;
  const int nk = K / BK;
  int best = 0;
  for (int S = 2; S <= 32; S *= 2) {
    if (nk % (2 * S) || (size_t)S * M * N * 4 > ws_bytes) break;
    best = S;
    if (tiles * S >= 256) break;                           // one block per CU reached
  }
  return best;
}

// ---- Which path takes a product that all of them could: the least estimated time.
enum Route { ROUTE_NONE, ROUTE_SKINNY, ROUTE_SPLIT, ROUTE_MID, ROUTE_128, ROUTE_192, ROUTE_256, ROUTE_V11 };

// The blocks that the mid-M path takes.
enum MidForm { MID_16, MID_16X2, MID_32, MID_64, MID_64_W4, MID_128R, MID_128, MID_128_W4 };
// Blocks of 16 pairs, or of two 16-column panels, for up to 64 rows.  Up to a round of them the mid blocks leave half of the CUs idle
// (plain products of up to 128: the 16-column blocks fill them).  Above it, up to 16 rows (plain ones to 32), the mid blocks have the
// 64-row tile's staging of A to carry, but few K-tiles, or two rounds of the mid blocks that end together (768 .. 1,024), are as fast
// there (0.98 to 1.27), and with more rows everything above a round is (1.0 to 1.4).  Random products that this rule gives them: 672 pairs
// 0.70 of the mid blocks' time (worst 1.02), plain ones 0.62 to 0.87 up to a round, 0.83 to 0.95 above.
bool two_panels(int M, int N, int K, bool pairs) {
  const int b = N / 32;
  if (b <= 256) return pairs || b > 128;
  if (!pairs && M <= 32 && K >= 2560 && b <= 768) return true;
  return M <= 16 && K >= 1024 && (b <= 512 || (K >= 1280 && b <= 768) || (b > 1024 && (pairs || K >= 2048)));
}
// pairs: an epilogue that joins columns (SwiGLU, RoPE).  panels: two-panel blocks among them.  K % 128 == 0
MidForm mid_form(int M, int N, int K, bool pairs, bool bn64_ok, bool panels = true) {
  // 64-column blocks for a single row tile whose 128-column grid fills less than one round of the
  // 256 CUs: 70B generation steps with 8 prompts (M = 40) 39.7 vs 46.7 ms per step; with 32 prompts
  // (M = 160, three row tiles) the 128-column blocks are faster, 53 vs 55.5 ms (profiles/r6_decode/
  // mid_bn: in-graph steps, cold weights; a same-weights GEMM loop favoured 64 there too)
  const int tiles_m = (M + mid::BMm - 1) / mid::BMm;
  const int blocks128 = tiles_m * (N / mid::BNm);
  // (and, since the 8-wave blocks, for two row tiles of at most ~1.25 rounds: 70B at M = 96, down
  // 193 -> 147 us, O 49 -> 36 us; profiles/r6_decode/mid8/bn64_m96_gemm_bench.log)
  const int blocks64 = tiles_m * (N / 64);
  const bool bn64 = bn64_ok && (g_mid_bn == 64 || (g_mid_bn == 0 && ((blocks128 < 256 && M <= mid::BMm) ||
                                                                     (M <= 2 * mid::BMm && blocks64 <= 320))));
  // 8 waves for grids of < 2 rounds of 64-row blocks; 128-row blocks when 64-row ones take more than
  // one round, 128-row ones fit in one and K is long (profiles/r6_decode/mid8, 70B at M = 320: down
  // 343 -> 276 us; the K = 8,192 projections ran 5-10% slower with 128 rows)
  const bool w8 = g_mid_waves == 8 || (g_mid_waves == 0 && blocks128 < 512);
  const int rows128 = (M + 127) / 128 * (N / mid::BNm);
  const bool r128 = g_mid_rows == 128 || (g_mid_rows == 0 && blocks128 > 256 && rows128 <= 256 && K >= 16384);
  const bool w8_64 = g_mid_waves == 8 || (g_mid_waves == 0 && blocks64 < 512);
  // 32-column blocks (NONE / RESID epilogues) when even 64-column ones leave CUs idle: the 70B O and
  // down projections of generation steps with <= 12 prompts (M <= 64: 128 -> 256 blocks)
  const bool bn32 = !pairs && N % 32 == 0 && g_mid_waves != 4 &&
                    (g_mid_bn == 32 || (g_mid_bn == 0 && M <= mid::BMm && blocks64 < 256));
  // 16-column ones where 32-column ones leave CUs idle too (g_mid_bn: a forced width keeps the mid blocks)
  const bool few = M <= mid::BMm && K % 256 == 0 && g_mid_waves != 4;
  if (panels && few && (g_mid_bn == 33 || (g_mid_bn == 16 && pairs) || (g_mid_bn == 0 && two_panels(M, N, K, pairs)))) return MID_16X2;
  if (few && !pairs && (g_mid_bn == 16 || (bn32 && g_mid_bn == 0 && N / 32 < 256))) return MID_16;
  if (bn32) return MID_32;
  if (bn64) return w8_64 ? MID_64 : MID_64_W4;
  if (w8) return r128 ? MID_128R : MID_128;
  return MID_128_W4;
}

// (The 64-column blocks take 0.92 of what is estimated for them since their K-tiles are of 128 terms.  Fitted anew they took products of
// 65 to 128 rows from K-split blocks, whose estimates are further off: 1.002 of the time of 180 random ones, up to 1.2, and 0.995, up to
// 1.04, with these.) The estimates (us).  Fitted to 15,400 random products of 1 .. 3,000 rows, 512 .. 29,440 columns (and a gate / up of
// 57,344) and 256 .. 28,928 terms, each timed on every path that it can take, with weights that no cache holds;
// profiles/cases/gemm_routes.txt has the errors of the fits, 5 to 9% each, and what the choice makes of them.  The shortest form that
// tells the paths apart: a start, and the larger of the weight's stream and the K tiles of 64 terms (nk), which take longer the more
// blocks pull on memory and power at once.
struct MidCost { float start, k_few, k_full, start2, k2, k2_more, tb; };       // tb: bytes of weight a us, in millions
const MidCost MID_16_COST[3] = {{4.7f, 0.05f, 0.152f, 7.4f, 0.199f, 0.f, 4.76f}, {5.f, 0.092f, 0.165f, 7.8f, 0.247f, 0.f, 4.97f},
                                {4.7f, 0.147f, 0.207f, 6.8f, 0.33f, 0.f, 4.99f}};        // up to 16, 32 and 64 rows
// (two panels: of 2,600 random products launch to launch in a graph, so that only SKINNY_COST's last compares with them; 5% off)
const MidCost MID_16X2_COST[3] = {{2.9f, 0.112f, 0.147f, 3.7f, 0.273f, 0.277f, 5.63f}, {3.f, 0.123f, 0.183f, 5.6f, 0.301f, 0.048f, 5.23f},
                                  {2.7f, 0.177f, 0.242f, 4.f, 0.27f, 0.13f, 5.2f}};
const MidCost MID_32_COST = {4.4f, 0.269f, 0.337f, 6.f, 0.415f, 0.f, 4.2f};
const MidCost MID_64_COST[2] = {{4.8f, 0.279f, 0.452f, 6.7f, 0.658f, 0.f, 4.8f}, {4.9f, 0.288f, 0.366f, 5.9f, 0.524f, 0.f, 5.f}};      // up to 64, 128 rows
const MidCost MID_128_COST[2] = {{7.f, 0.38f, 0.543f, 8.9f, 0.833f, 0.173f, 5.6f}, {5.5f, 0.387f, 0.476f, 7.8f, 0.65f, 0.235f, 5.f}};
const MidCost MID_128R_COST = {-14.f, 0.514f, 0.7f, 18.f, 0.6f, 0.3f, 3.8f};
float mid_us(int M, int N, int K, MidForm form) {
  const int tiles_m = (M + 63) / 64;
  const float nk = (float)(K / BK), bytes = (float)N * K * 2.f;
  const MidCost& c = form == MID_16 || form == MID_16X2 ? (form == MID_16 ? MID_16_COST : MID_16X2_COST)[M <= 16 ? 0 : M <= 32 ? 1 : 2]
                     : form == MID_32 ? MID_32_COST
                     : form == MID_64 || form == MID_64_W4 ? MID_64_COST[M > 64]
                     : form == MID_128R ? MID_128R_COST : MID_128_COST[M > 128];
  const int width = form == MID_16 ? 16 : form == MID_16X2 || form == MID_32 ? 32 : form == MID_64 || form == MID_64_W4 ? 64 : 128;
  const float rounds = (float)((form == MID_128R ? (M + 127) / 128 : tiles_m) * (N / width)) / 256.f;
  if (form == MID_128_W4) return (4.f + 0.532f * nk) * powf(rounds, 0.842f);
  if (rounds <= 1.f) return c.start + fmaxf(bytes / (c.tb * 1e6f), (c.k_few + (c.k_full - c.k_few) * rounds) * nk);
  // (two blocks of two panels share a CU: up to two rounds some CUs have both and take as long as all with both)
  const float more = form == MID_16X2 ? fmaxf(rounds - 2.f, 0.f) : rounds - 1.f;
  return c.start2 + fmaxf(bytes / (c.tb * 1e6f), (c.k2 + c.k2_more * more) * nk);
}

// Tiles of `rows` x 256: whole rounds of 256 blocks and a last one.  A weight that one or two row tiles read comes from memory and not from
// another block's read (alone).  Rounds are why no one tile serves a range: 600 x 12,288 x 4,096 on 256-row tiles is 144 blocks of 79 us, on
// 128-row ones 240 of 62; 600 x 22,016 258 blocks (two rounds, 168 us) or 430 (117).
struct RoundCost { int rows; float full_k, full, part_k, part, fill, alone; };
const RoundCost ROUNDS[4] = {{128, 0.798f, 9.3f, 0.406f, 5.8f, 0.148f, 0.305f}, {192, 1.006f, 12.2f, 0.704f, 9.4f, 0.609f, 0.18f},
                             {256, 1.311f, 14.1f, 0.91f, 11.5f, 0.979f, 0.074f}, {384, 1.907f, 17.7f, 1.458f, 14.7f, 1.17f, 0.119f}};
float rounds_us(const RoundCost& c, int M, int N, int K) {
  const int tiles_m = (M + c.rows - 1) / c.rows;
  const long blocks = (long)tiles_m * (N / BN);
  const float nk = (float)(K / BK) * (1.f + c.alone / (float)tiles_m);
  const float full = c.full_k * nk + c.full, part = c.part_k * nk + c.part, fill = (float)(blocks % 256) / 256.f;
  return (float)(blocks / 256) * full + (fill > 0.f ? part + (full - part) * powf(fill, c.fill) : 0.f);
}
// The same cut along K into S slices, and their sum
float split_us(int M, int N, int K, int S) {
  const int tiles_m = (M + 255) / 256;
  const long blocks = (long)tiles_m * (N / BN) * S;
  const float nk = (float)(K / BK) / S;
  const float full = 1.365f * nk + 3.2f, part = 0.822f * nk, fill = (float)(blocks % 256) / 256.f;
  const float tiles = (float)(blocks / 256) * full + (fill > 0.f ? part + (full - part) * powf(fill, 0.349f) : 0.f);
  return 12.2f + fmaxf((float)N * K * 2.f / 4.04e6f, tiles) + S * ((float)M * N * 1.314e-6f + 0.094f);
}
// K-split blocks of all rows (gemm_skinny.h): up to 64 rows, more without a split, more; up to 64 beside blocks of two panels, timed as those
struct SkinnyCost { float start, tb, k, k_rows, k_fill, over, slab, slice, sum; };
const SkinnyCost SKINNY_COST[4] = {{4.9f, 4.48f, 0.2f, 0.1115f, 0.408f, 1.097f, 2.19f, 0.41f, 2.4f}, {7.f, 4.94f, -0.15f, 0.167f, 0.785f, 1.f, 0.f, 0.f, 0.f},
                                   {0.f, 4.55f, 0.194f, 0.0955f, 0.231f, 1.167f, 1.73f, 0.17f, 9.5f}, {2.3f, 5.81f, 0.246f, 0.09f, 0.262f, 1.174f, 1.73f, 0.49f, 1.7f}};
float skinny_us(int M, int N, int K, int bn, int S, bool beside_panels = false) {
  const SkinnyCost& c = SKINNY_COST[beside_panels ? 3 : M <= 64 ? 0 : S == 1 ? 1 : 2];
  const float rounds = (float)(N / bn) * S / 256.f;
  const float k = (c.k + c.k_rows * ((M + 31) / 32) + c.k_fill * fminf(rounds, 1.f)) * powf(fmaxf(rounds, 1.f), c.over);
  return c.start + fmaxf((float)N * K * 2.f / (c.tb * 1e6f), k * (float)(K / BK) / S) +
         (S > 1 ? c.sum + S * (c.slab * (float)M * N * 1e-6f + c.slice) : 0.f);
}

// The rules by shape alone, for what the estimates do not serve (launch, ROUTE_NONE)
bool split_rule(int M, size_t tiles256, int S) { return S >= 2 && (M > 64 || tiles256 * S >= 128); }
bool mid_rule(int M, size_t tiles256) { return tiles256 < 128 || (M <= 64 && tiles256 < 512); }

// ws: scratch for split-K partials (0 bytes: none).  Above four rounds of 256-row tiles the forms are within 3% of each other:
// ROUTE_NONE (v11 or v10 by whole rounds, v11_pays).  A path that the rules by shape take keeps the product unless another is estimated more
// than 6% faster, which is how far off the estimates are: of 13,900 products 0.5% are then more than 6% slower than by the rules, and all
// take 0.86 of their time by the rules, 1.005 of the best path's.
Route route_of(int M, int N, int K, int epi, bool row_exact, size_t ws_bytes) {
  const long tiles256 = (long)((M + 255) / 256) * (N / BN);
  if (M > ROW_CHUNK || tiles256 > 1024 || g_v10_rows || g_mid_bn || g_mid_waves || g_mid_rows || g_skinny > 1) return ROUTE_NONE;
  if (M <= 64 && (row_exact || !g_mid || !g_skinny)) return ROUTE_NONE;
  const bool pairs = epi == FLS_EPI_SWIGLU || is_rope(epi);
  const bool scratch = !row_exact && ws_bytes > 0;
  const int bn = skinny_bn(M, N, K), S = skinny_slices(N, K, bn);
  const bool skinny = !row_exact && g_skinny && M <= 256 && (S == 1 || (size_t)S * M * N * 4 <= ws_bytes) && (M > 32 ? M > 64 || !skinny_wide(N) : true);
  const int S2 = scratch && g_splitk && M > 64 && M <= SPLITK_MAX_M ? splitk_slices(M, N, K, (size_t)tiles256, ws_bytes) : 0;
  const bool split = split_rule(M, (size_t)tiles256, S2);
  const Route rules = skinny && skinny_range(M, N) ? ROUTE_SKINNY
                      : split ? ROUTE_SPLIT
                      : g_mid && mid_rule(M, (size_t)tiles256) ? ROUTE_MID
                      : M >= 384 && (long)((M + 383) / 384) * (N / BN) >= 256 && fls_gemm_v11_pays(M, N) ? ROUTE_V11 : ROUTE_256;
  Route best = ROUTE_NONE;
  float least = 0.f;
  auto offer = [&](Route r, float us) {
    if (r == rules) us *= 0.94f;
    if (best == ROUTE_NONE || us < least) {
      best = r;
      least = us;
    }
  };
  if (g_mid) offer(ROUTE_MID, mid_us(M, N, K, mid_form(M, N, K, pairs, true, false)));
  if (skinny) offer(ROUTE_SKINNY, skinny_us(M, N, K, bn, S));
  if (split) offer(ROUTE_SPLIT, split_us(M, N, K, S2));
  if (M > 64) {              // (up to 64 rows one row tile covers them all, and three quarters of a 256-row one are padding)
    for (int i = 0; i < 3; ++i) offer((Route)(ROUTE_128 + i), rounds_us(ROUNDS[i], M, N, K));
    if (M >= 384) offer(ROUTE_V11, rounds_us(ROUNDS[3], M, N, K));
  } else if (best == ROUTE_SKINNY && mid_form(M, N, K, pairs, true) == MID_16X2 &&
             1.04f * mid_us(M, N, K, MID_16X2) < skinny_us(M, N, K, bn, S, true)) {
    // Two panels take what the mid blocks would, and of the K-split blocks' products those that they are estimated 4% faster for.  2,600
    // random ones of up to 64 rows, against the time before there were two panels: 0.896, 6 of them more than 5% slower (no margin: 0.894,
    // 32; each on the faster of the two: 0.890)
    best = ROUTE_MID;
  }
  return best;
}

// what launch returns where the product has also written the K/V rows (Epi::kv_dst): no error code of HIP's
constexpr int KV_WRITTEN = 1 << 24;

// -> 0, KV_WRITTEN, or an error
template <int EPI>
int launch(const half_t* A, const half_t* W, half_t* C, int M, int N, int K, int lda, int ldw, int ldc,
           const Epi& ep, hipStream_t s, void* ws, size_t ws_bytes, Route route) {
  const bool mid_ok = N % mid::BNm == 0 && K % mid::BKm == 0 && lda % 8 == 0 && ldw % 8 == 0;
  const size_t tiles256 = (size_t)((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  // 32-bit per-lane DMA offsets (X rows; SWIGLU up-block rows)
  const bool offs32 = (size_t)M * lda * 2 < (1ull << 32) &&
                      (EPI != FLS_EPI_SWIGLU || (size_t)(N / 2 + BN) * ldw * 2 < (1ull << 32));
  // the v10 epilogues store (and load the residual) 16 B per lane
  const bool wide_ok = ldc % 8 == 0 && ((uintptr_t)C & 15) == 0 &&
                       (EPI != FLS_EPI_RESID || (ep.ldr % 8 == 0 && ((uintptr_t)ep.R & 15) == 0));
  const bool main_ok = N % BN == 0 && K % BK == 0 && (K / BK) % 2 == 0 && lda % 8 == 0 && ldw % 8 == 0 && offs32 &&
                       wide_ok;
  // Too few 256x256 tiles for 256 CUs -> 64x128 tiles.  Measured crossover (profiles/r1_gemm_mid):
  // the mid kernel wins below ~128 main tiles, and at M <= 64 (3/4 of every 256-row tile wasted)
  // up to 512; above that its lower L2 reuse (43 vs 128 FLOP per staged byte) costs more than the
  // idle CUs.  It is also the path for odd K-tile counts.
  // split-K for small M: the whole weight read once, every CU streaming (see splitk_reduce_kernel)
  const bool split_ok = g_splitk && ws && M <= SPLITK_MAX_M && N % BN == 0 && K % BK == 0 && lda % 8 == 0 &&
                        ldw % 8 == 0 && (size_t)M * lda * 2 < (1ull << 32) && ldc % 4 == 0 &&
                        ((uintptr_t)C & 7) == 0 && ((uintptr_t)ws & 15) == 0 &&
                        (EPI != FLS_EPI_RESID || (ep.ldr % 4 == 0 && ((uintptr_t)ep.R & 7) == 0));
  if (!main_ok) route = ROUTE_NONE;
  // The row statistic of A (rs_eps): made by the blocks of 16 pairs where they take the product, have waves for it and registers for its
  // parts, else by a launch here.
  constexpr bool pairs = EPI != FLS_EPI_NONE && EPI != FLS_EPI_RESID;
  const bool to_mid = mid_ok && (ep.row_exact || route == ROUTE_MID) &&
                      (!main_ok || route == ROUTE_MID || (route == ROUTE_NONE && g_mid && mid_rule(M, tiles256)));
  const bool bn64_ok = N % 64 == 0 && (EPI != FLS_EPI_ROPE || N % 128 == 0);
  const bool stat = ep.rs_eps > 0.f && pairs && to_mid && M <= 32 && K <= 8192 && mid_form(M, N, K, pairs, bn64_ok) == MID_16X2;
  if (ep.rs_eps > 0.f && !stat) row_stat(A, lda, M, K, ep.rs_eps, const_cast<float*>(ep.rs), s);
  if (!ep.row_exact && (route == ROUTE_NONE || route == ROUTE_SKINNY)) {
    const int rc = try_skinny<EPI>(A, W, C, M, N, K, lda, ldw, ldc, ep, s, ws, ws_bytes, route == ROUTE_SKINNY);
    if (rc > 0) ss_partials(C, ldc, M, N, ep, s);
    if (rc) return rc > 0 ? 0 : rc;
  }
  if (route == ROUTE_SKINNY) route = ROUTE_NONE;             // (its operands' alignment did not allow it)
  const int S = split_ok && !ep.row_exact && (route == ROUTE_NONE || route == ROUTE_SPLIT)
                    ? splitk_slices(M, N, K, tiles256, ws_bytes) : 0;
  if (split_rule(M, tiles256, S)) {
    static bool attr_f32 = false;
    if (!attr_f32) {
      (void)hipFuncSetAttribute((const void*)gemm_nt_v10<EPI_F32>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                2 * BUF);
      attr_f32 = true;
    }
    Epi e = ep;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = N / BN;
    e.order = g_order ? g_order : auto_order(tiles_m, tiles_n);
    e.ksplit = S;
    e.kslice = K / S;
    e.part_stride = (long long)M * N;
    float* part = (float*)ws;
    hipLaunchKernelGGL((gemm_nt_v10<EPI_F32>), dim3((int)tiles256 * S), dim3(256), 2 * BUF, s, A, W, (half_t*)part, M,
                       N, K / S, lda, ldw, N, e);
    FLS_CHECK_LAUNCH();
    const long long threads = (long long)M * (N / 4);
    hipLaunchKernelGGL(splitk_reduce_kernel<EPI>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, part, S,
                       e.part_stride, M, N, C, ldc, e);
    FLS_CHECK_LAUNCH();
    ss_partials(C, ldc, M, N, ep, s);
    FLS_CHECK_LAUNCH();
    return 0;
  }
  if (route == ROUTE_SPLIT) route = ROUTE_NONE;
  if (mid_ok && (!main_ok || route == ROUTE_MID ||
                 (route == ROUTE_NONE && g_mid && mid_rule(M, tiles256)))) {
    bool kv_written = false;
    switch (mid_form(M, N, K, pairs, bn64_ok)) {
      case MID_16:
        if constexpr (!pairs) {
          if (M <= 16) launch_col16<EPI, 1, 1>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
          else if (M <= 32) launch_col16<EPI, 2, 1>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
          else launch_col16<EPI, 4, 1>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
        }
        break;
      case MID_16X2:
        kv_written = is_rope(EPI) && ep.kv_dst != nullptr;
        if constexpr (pairs) {
          if (stat) {
            if (M <= 16) launch_col16<EPI, 1, 2, true>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
            else launch_col16<EPI, 2, 2, true>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
            break;
          }
        }
        if (M <= 16) launch_col16<EPI, 1, 2>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
        else if (M <= 32) launch_col16<EPI, 2, 2>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
        else launch_col16<EPI, 4, 2>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
        break;
      case MID_32:
        if constexpr (!pairs) launch_mid<EPI, mid::NSTAGE, 32, 8>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
        break;
      case MID_64:
        if (K % 128) launch_mid<EPI, 4, 64, 8>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
        else if ((M + 63) / 64 * (N / 64) <= 256) launch_mid<EPI, 3, 64, 8, 64, 128>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
        else launch_mid<EPI, 2, 64, 8, 64, 128>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
        break;
      case MID_64_W4: launch_mid<EPI, mid::NSTAGE, 64>(A, W, C, M, N, K, lda, ldw, ldc, ep, s); break;
      case MID_128R: launch_mid<EPI, mid::NSTAGE, 128, 8, 128>(A, W, C, M, N, K, lda, ldw, ldc, ep, s); break;
      case MID_128:
        if (K % 128 == 0 && K >= 2048 && (M + 63) / 64 * (N / 128) <= 256) launch_mid<EPI, 3, 128, 8, 64, 128>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
        else launch_mid<EPI, mid::NSTAGE, 128, 8>(A, W, C, M, N, K, lda, ldw, ldc, ep, s);
        break;
      case MID_128_W4: launch_mid<EPI, mid::NSTAGE, 128>(A, W, C, M, N, K, lda, ldw, ldc, ep, s); break;
    }
    FLS_CHECK_LAUNCH();
    ss_partials(C, ldc, M, N, ep, s);
    FLS_CHECK_LAUNCH();
    return kv_written ? KV_WRITTEN : 0;
  }
  if (!main_ok) {
    dim3 grid((M + 31) / 32, (N + 255) / 256);
    hipLaunchKernelGGL(gemm_nt_generic<EPI>, grid, dim3(256), 0, s, A, W, C, M, N, K, lda, ldw, ldc, ep);
    FLS_CHECK_LAUNCH();
    ss_partials(C, ldc, M, N, ep, s);
    FLS_CHECK_LAUNCH();
    return 0;
  }
  // Row chunks of <= ROW_CHUNK rows: with more rows the activation panel (M x K) outgrows the 256 MB
  // Infinity Cache and the N-grouped tile order re-reads it from HBM once per group of weight
  // columns.  70B O projection over 43,008 rows: one launch 1,361 TFLOP/s, three of 14,336 rows
  // 1,421 (gate/up + SwiGLU 1,325 -> 1,430; profiles/r3_gemm, scripts/gemm_m_chunks.py).
  // Only when every chunk still fills the chip (>= 256 tiles), so each piece stays on this path.
  const int n_chunks = (M + ROW_CHUNK - 1) / ROW_CHUNK;
  const int step = ((M + n_chunks - 1) / n_chunks + BM - 1) / BM * BM;
  if (route <= ROUTE_MID && M > ROW_CHUNK && (size_t)(step / BM) * (N / BN) >= 256) {
    for (int r0 = 0; r0 < M; r0 += step) {
      Epi e = ep;
      if (e.pos) e.pos += r0;
      if (e.R) e.R += (size_t)r0 * e.ldr;
      if (e.ss) e.ss += (size_t)r0 * e.ss_ld;
      if (e.rs) e.rs += r0;                  // (the fused norm's per-row statistic follows its rows)
      const int rc = launch<EPI>(A + (size_t)r0 * lda, W, C + (size_t)r0 * ldc, min(step, M - r0), N, K, lda, ldw,
                                 ldc, e, s, ws, ws_bytes, ROUTE_NONE);
      if (rc) return rc;
    }
    return 0;
  }
  // One block per tile, dispatched by the hardware as CUs free up.  A persistent form (one block
  // per CU walking its tiles, the next tile's prologue DMA under this tile's epilogue) measured
  // 1.1-3.9% slower on every 70B / 7B shape once the tile order was XCD-aware (profiles/r2_gemm).
  launch_main<EPI>(g_v10_rows ? g_v10_rows : route == ROUTE_128 ? 128 : route == ROUTE_192 ? 192 : 256, A, W, C, M, N, K, lda, ldw, ldc, ep, s);
  FLS_CHECK_LAUNCH();
  return 0;
}

}  // namespace

extern "C" int fls_kernels_version(void) { return 40; }

// tile order: 0 = by shape (default); g > 0: groups of g M tiles; g < 0: groups of -g N tiles (A/B, tests)
extern "C" int fls_gemm_set_order(int order) {
  const int old = g_order;
  g_order = order;
  return old;
}

// skinny-M path (gemm_skinny.h): 0 off, 1 auto (default), 2 every M <= 256 it supports; blocks: the
// K-split block target (0: the whole-round rule, the default); returns the previous mode
extern "C" int fls_gemm_set_skinny(int mode, int blocks) {
  const int old = g_skinny;
  g_skinny = mode < 0 ? 0 : mode > 2 ? 2 : mode;
  g_skinny_blocks = blocks > 0 ? blocks : 0;
  return old;
}

// skinny-M weight rows per block: 0 auto (default), 128 or 256 where supported; returns the previous
extern "C" int fls_gemm_set_skinny_bn(int bn) {
  const int old = g_skinny_bn;
  g_skinny_bn = bn == 128 || bn == 256 ? bn : 0;
  return old;
}

// split-K path for small M on (1, default) or off (0; tests / A-B)
extern "C" int fls_gemm_set_splitk(int on) {
  const int old = g_splitk;
  g_splitk = on ? 1 : 0;
  return old;
}

// rows of a v10 tile: 0 by shape (default), 128, 192 or 256 forced (tests / A-B); returns the previous
extern "C" int fls_gemm_set_v10_rows(int rows) {
  const int old = g_v10_rows;
  g_v10_rows = rows == 128 || rows == 192 || rows == 256 ? rows : 0;
  return old;
}

// rows per main-path launch (0: unlimited; default 16384)
extern "C" int fls_gemm_set_row_chunk(int rows) {
  const int old = ROW_CHUNK;
  ROW_CHUNK = rows > 0 ? rows : (1 << 30);
  return old;
}

// per-row partial sums of squares of an fp16 [rows, H] matrix, one fp32 per 128 columns (H % 128 == 0):
// the residual GEMM epilogue's partials, bitwise, for a hidden state that arrived without them
extern "C" int fls_row_ss(const void* x, int ldx, int rows, int H, float* ss, int ss_ld, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (H % 128 || ldx % 4 || ((uintptr_t)x & 7) || ss_ld < H / 128) return -2;
  ss_partials_raw((const half_t*)x, ldx, rows, H, ss, ss_ld, (hipStream_t)s);
  FLS_CHECK_LAUNCH();
  return 0;
}

// rstd[r] = rsqrt(mean(x[r]^2) + eps) for an fp16 [rows, H] matrix (H % 128 == 0, H <= 16,384), bitwise
// fls_row_ss + fls_rstd_from_ss (the fused norm's statistic without a residual GEMM's partials)
extern "C" int fls_row_stat(const void* x, int ldx, int rows, int H, float eps, float* rstd, fls_stream_t s) {
  if (rows <= 0) return 0;
  if (H % 128 || H / 128 > ROW_STAT_MAX_PARTS || ldx % 8 || ((uintptr_t)x & 15)) return -2;
  row_stat((const half_t*)x, ldx, rows, H, eps, rstd, (hipStream_t)s);
  FLS_CHECK_LAUNCH();
  return 0;
}

// mid-M block columns: 0 auto (default), 16 (M <= 64), 32, 64 or 128 forced where valid (tests / A-B; 32: NONE / RESID
// epilogues, 8 waves; 16: two panels where the epilogue joins columns; 33: two panels); returns the previous
extern "C" int fls_gemm_set_mid_bn(int bn) {
  const int old = g_mid_bn;
  g_mid_bn = bn == 16 || bn == 33 || bn == 32 || bn == 64 || bn == 128 ? bn : 0;
  return old;
}

// 128-column mid-M blocks: 0 auto (default: 8 waves for grids of < 512 blocks), 4 or 8 waves forced
// (tests / A-B); returns the previous
extern "C" int fls_gemm_set_mid_waves(int waves) {
  const int old = g_mid_waves;
  g_mid_waves = waves == 4 || waves == 8 ? waves : 0;
  return old;
}

// 8-wave mid-M blocks' rows: 0 auto (default: 128 when 64-row blocks would take more than one round
// and 128-row ones fit in one), 64 or 128 forced (tests / A-B); returns the previous
extern "C" int fls_gemm_set_mid_rows(int rows) {
  const int old = g_mid_rows;
  g_mid_rows = rows == 64 || rows == 128 ? rows : 0;
  return old;
}

// mid-M kernel for small grids on (1, default) or off (0; tests)
extern "C" int fls_gemm_set_mid(int on) {
  const int old = g_mid;
  g_mid = on ? 1 : 0;
  return old;
}

// gemm_v11.hip: the 384 x 256 tile for large projections (returns 1 when it took the GEMM)
extern "C" int fls_gemm_v11_try(const void* A, const void* W, void* C, const void* R, int M, int N, int K, int lda,
                                int ldw, int ldc, int ldr, int epi, const int* pos, const float* cos_t,
                                const float* sin_t, int rope_cols, int head_dim, const void* bias,
                                const float* rscale, float alpha, float* ss, int ss_ld, int want, fls_stream_t s);

// Does a residual product of M x N x K write its rows' partial sums of squares in its epilogue (v10 and v11 tiles)?  On the other paths
// they are a launch of their own behind it and a second one sums them; fls_row_stat gives the same bits in one (79 rows x 4,096:
// 3.5 + 2.7 us and a launch more, 2.6 here).
extern "C" int fls_gemm_leaves_ss(int M, int N, int K, uint64_t ws_bytes) {
  if (M <= 64 || N % BN || K % (2 * BK)) return 0;
  const Route route = route_of(M, N, K, FLS_EPI_RESID, false, ws_bytes);
  return route == ROUTE_NONE ? (long)((M + 255) / 256) * (N / BN) >= 128 : route >= ROUTE_128;
}

namespace {
struct KvOut {
  half_t* kv;
  half_t* const* kv_at;
  const int* dst;
  int col0, ld;
};
// fls_gemm; KV_WRITTEN where the product has also written the K/V rows
int gemm_entry(const void* A, const void* W, void* C, const void* R, int M, int N, int K, int lda, int ldw,
               int ldc, int ldr, int epi, const int* pos, const float* cos_t, const float* sin_t,
               int rope_cols, int head_dim, const void* bias, const float* rscale, float rs_eps, float alpha, float* ss,
               int ss_ld, const KvOut* kv, void* ws, uint64_t ws_bytes, fls_stream_t s) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int row_exact = (epi & FLS_GEMM_ROW_EXACT) ? 1 : 0;
  epi &= 0xff;
  // row partial sums of squares: residual GEMMs only, one per 128 output columns
  if (ss && (epi != FLS_EPI_RESID || N % 128 || ss_ld < N / 128)) return -7;
  if (bias && epi == FLS_EPI_SWIGLU) return -4;
  if ((epi == FLS_EPI_SWIGLU || epi == FLS_EPI_ROPE) && (N % 32)) return -2;
  if (epi == FLS_EPI_ROPE && ((head_dim != 64 && head_dim != 128) || rope_cols % head_dim || N % head_dim))
    return -3;
  // rscale made here: by the path itself or by fls_row_stat's kernel in front of it
  if (rs_eps > 0.f) {
    if (!rscale || K % 128 || K / 128 > ROW_STAT_MAX_PARTS || lda % 8 || ((uintptr_t)A & 15)) return -2;
    if (M > 64) {
      row_stat((const half_t*)A, lda, M, K, rs_eps, const_cast<float*>(rscale), (hipStream_t)s);
      rs_eps = 0.f;
    }
  }
  Route route = N % BN == 0 && K % (2 * BK) == 0 ? route_of(M, N, K, epi, row_exact != 0, ws ? ws_bytes : 0) : ROUTE_NONE;
  if (M > 64) {
    const int rc = fls_gemm_v11_try(A, W, C, R, M, N, K, lda, ldw, ldc, ldr, epi, pos, cos_t, sin_t, rope_cols,
                                    head_dim, bias, rscale, alpha, ss, ss_ld,
                                    route == ROUTE_NONE ? 0 : route == ROUTE_V11 ? 1 : -1, s);
    if (rc) return rc > 0 ? 0 : rc;
    if (route == ROUTE_V11) route = ROUTE_NONE;
  }
  Epi ep{(const half_t*)R, ldr, pos, cos_t, sin_t, rope_cols, head_dim, (const half_t*)bias, N / 2, 0,
         nullptr, nullptr, 0, 0};
  ep.rs = rscale;
  ep.rs_eps = rs_eps;
  if (kv != nullptr) {
    ep.kv = kv->kv;
    ep.kv_at = kv->kv_at;
    ep.kv_dst = kv->dst;
    ep.kv_col0 = kv->col0;
    ep.kv_ld = kv->ld;
  }
  ep.alpha = alpha;
  ep.ss = ss;
  ep.ss_ld = ss_ld;
  ep.row_exact = row_exact;
  auto a = (const half_t*)A;
  auto w = (const half_t*)W;
  auto c = (half_t*)C;
  auto st = (hipStream_t)s;
  switch (epi) {
    case FLS_EPI_NONE: return launch<FLS_EPI_NONE>(a, w, c, M, N, K, lda, ldw, ldc, ep, st, ws, ws_bytes, route);
    case FLS_EPI_RESID: return launch<FLS_EPI_RESID>(a, w, c, M, N, K, lda, ldw, ldc, ep, st, ws, ws_bytes, route);
    case FLS_EPI_SWIGLU: return launch<FLS_EPI_SWIGLU>(a, w, c, M, N, K, lda, ldw, ldc, ep, st, ws, ws_bytes, route);
    case FLS_EPI_ROPE:
      return head_dim == 128 ? launch<FLS_EPI_ROPE>(a, w, c, M, N, K, lda, ldw, ldc, ep, st, ws, ws_bytes, route)
                             : launch<EPI_ROPE64>(a, w, c, M, N, K, lda, ldw, ldc, ep, st, ws, ws_bytes, route);
  }
  return -1;
}
}  // namespace

extern "C" int fls_gemm(const void* A, const void* W, void* C, const void* R, int M, int N, int K, int lda, int ldw,
                        int ldc, int ldr, int epi, const int* pos, const float* cos_t, const float* sin_t,
                        int rope_cols, int head_dim, const void* bias, const float* rscale, float rs_eps, float alpha, float* ss,
                        int ss_ld, void* ws, uint64_t ws_bytes, fls_stream_t s) {
  return gemm_entry(A, W, C, R, M, N, K, lda, ldw, ldc, ldr, epi, pos, cos_t, sin_t, rope_cols, head_dim, bias, rscale, rs_eps, alpha, ss, ss_ld, nullptr, ws,
                    ws_bytes, s);
}

// A RoPE product whose rows' columns from kv_col0 on (new keys and values) also go to rows kv_dst of a K/V buffer: from the blocks of 16 pairs with
// their own stores, else by fls_copy_rows behind it (16 rows x 8,192 columns: 4.6 us and a launch of a generation step's layer)
extern "C" int fls_gemm_kv(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, int epi, const int* pos, const float* cos_t,
                           const float* sin_t, int rope_cols, int head_dim, const void* bias, const float* rscale, float rs_eps, void* kv, void* const* kv_at,
                           const int* kv_dst, int kv_col0, int kv_ld, void* ws, uint64_t ws_bytes, fls_stream_t s) {
  if (M <= 0) return 0;
  if ((epi & 0xff) != FLS_EPI_ROPE || !kv_dst || kv_col0 < 0 || kv_col0 >= N || kv_col0 % 8 || (head_dim > 0 && kv_col0 % head_dim) || kv_ld % 8 || ldc % 8 || N % 8 ||
      (kv_at == nullptr && (!kv || ((uintptr_t)kv & 15))) || ((uintptr_t)C & 15))
    return -2;
  const KvOut out = {(half_t*)kv, (half_t* const*)kv_at, kv_dst, kv_col0, kv_ld};
  const int rc = gemm_entry(A, W, C, C, M, N, K, lda, ldw, ldc, ldc, epi, pos, cos_t, sin_t, rope_cols, head_dim, bias, rscale, rs_eps, 1.f, nullptr, 0, &out, ws,
                            ws_bytes, s);
  if (rc) return rc == KV_WRITTEN ? 0 : rc;
  return fls_copy_rows((const half_t*)C + kv_col0, ldc, nullptr, kv, kv_ld, kv_at, kv_dst, M, N - kv_col0, s);
}
