// C[M,N] = epilogue(A[M,K] . W[N,K]^T), fp32 accumulation: the prompt projections of the stateful models.
//
// Both operands go from global memory to LDS by DMA (no registers in between), 128 bytes of a row at a time, 1 KiB pieces of
// 8 rows x 128 bytes whose 16-byte chunks are XOR-swizzled by the row (chunk c of row r in slot c ^ (r & 7)), so that the
// 16-byte fragment reads of 16x16x32 MFMAs have no bank conflicts.  Rows past M and columns past N re-read the last valid row
// (never out of bounds) and are not stored.
#include "seq_common.h"
#include "fls_seq.h"
#include "gemm_epi.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
#define LDS_AS __attribute__((address_space(3)))

struct Tile {
  const char* A;
  const char* W;
  void* C;
  Epi epi;
  int M, N, nk, lda, ldw, ldc;  // nk: K tiles; lda, ldw: bytes; ldc: elements
  const int* a_rows;        // row r of the product is made from row a_rows[r] of A (null: r)
  const int* offs;          // row groups (experts): group g owns rows offs[g] .. offs[g + 1] and weight g
  int groups;
  long long w_gs, a_gs, c_gs;   // group g's operands (bytes); strided batch (grid y): its columns of C (elements)
  int a_mod;
  int tiles_m, tiles_n, order;
  int ragged;               // columns or rows of C that four-column stores don't fit
};

// Virtual tile id -> (tile row, tile column): groups of `order` tiles of one dimension (order < 0: of N) walked along the
// other; with consecutive ids on one XCD, an XCD's concurrent tiles are a compact patch whose operand panels its L2 holds.
__device__ __forceinline__ int2 place(int b, int tiles_m, int tiles_n, int order) {
  const bool by_m = order > 0;
  const int g = by_m ? order : -order;
  const int along = by_m ? tiles_n : tiles_m, total = by_m ? tiles_m : tiles_n;
  const int first = b / (g * along) * g;
  const int size = min(total - first, g);
  const int in = b - first * along;
  const int grouped = first + in % size, walked = in / size;
  return by_m ? int2{grouped, walked} : int2{walked, grouped};
}

// An address that is the same in every lane, for a descriptor in scalar registers.  (Descriptors must be scalar: from a vector register each
// DMA is a loop over the lanes' descriptors.  So is one whose record count is a choice between -1 and 0, which is made as a vector sign
// extension; 1024 x 2048 x 2048 on 64 x 128 tiles 18.4 us with such loops, 15.5 without, 8448 x 2048 x 2048 on 128 x 128 97 and 81.)
__device__ __forceinline__ const char* uniform(const char* p) {
  const unsigned long long v = (unsigned long long)p;
  return (const char*)((unsigned long long)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 | (unsigned)__builtin_amdgcn_readfirstlane((int)v));
}

// This block's tile: rows [m0, mend) and first column of C, operands moved to its group; false: nothing to do.
template <int TM, int TN>
__device__ __forceinline__ bool locate(const Tile& a, const char*& A, const char*& W, size_t& cbase, int& m0, int& mend, int& n0) {
  int nwg = gridDim.x, tiles_m = a.tiles_m;
  int bid = blockIdx.x;
  // The launch covers the most tiles that row groups can have; only those there are take part, or whole XCDs get few or none (19384
  // rows at most, 15500 in 8 groups, 2 x 2048 columns, 2048 terms: 333 -> 274 us).
  if (a.offs != nullptr) {
    const int lane = threadIdx.x & 63;
    int cnt = 0;
    for (int g = lane; g < a.groups; g += 64) cnt += (a.offs[g + 1] - a.offs[g] + TM - 1) / TM;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
    tiles_m = __builtin_amdgcn_readfirstlane(cnt);
    nwg = tiles_m * a.tiles_n;
    if (bid >= nwg) return false;
  }
  {                                      // blocks go to the 8 XCDs in turn: give each a run of consecutive ids
    const int q = nwg >> 3, r = nwg & 7, xcd = bid & 7, loc = bid >> 3;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + loc;
  }
  const int2 t = place(bid, tiles_m, a.tiles_n, a.order);
  int tm = t.x;
  A = a.A;
  W = a.W;
  cbase = 0;
  mend = a.M;
  n0 = t.y * TN;
  m0 = 0;
  if (a.offs != nullptr) {               // tiles of the groups one after the other: find the one that owns tile tm
    const int lane = threadIdx.x & 63;
    int e = -1;
    for (int base = 0; base < a.groups; base += 64) {
      const int g = base + lane;
      const int cnt = g < a.groups ? (a.offs[g + 1] - a.offs[g] + TM - 1) / TM : 0;
      int pre = cnt;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(pre, o, 64);
        if (lane >= o) pre += v;
      }
      const unsigned long long past = __ballot(pre > tm);
      if (past != 0) {
        const int l = __builtin_ctzll(past);
        e = base + l;
        tm -= __shfl(pre, l, 64) - __shfl(cnt, l, 64);
        break;
      }
      tm -= __shfl(pre, 63, 64);
    }
    if (e < 0) return false;
    e = __builtin_amdgcn_readfirstlane(e);
    tm = __builtin_amdgcn_readfirstlane(tm);
    m0 = a.offs[e];
    mend = a.offs[e + 1];
    W += (size_t)e * a.w_gs;
  } else if (gridDim.y > 1) {
    const int g = blockIdx.y;
    A += (size_t)(g % a.a_mod) * a.a_gs;
    W += (size_t)g * a.w_gs;
    cbase = (size_t)g * a.c_gs;
  }
  m0 += tm * TM;
  return true;
}

// Byte offsets of a tile's row r of A (from row m0, or from the first row with a_rows) and of its row j of W.  Rows past
// the end re-read the last one.  A gated product takes 16 gate rows, their 16 up rows, the next 16 gate rows, ..., so that a wave
// has both halves of a column; its W is addressed from column n0 / 2 of the gate rows.
__device__ __forceinline__ unsigned a_offset(const Tile& a, int m0, int mend, int r) {
  r = min(r, mend - 1 - m0);
  return (unsigned)((a.a_rows != nullptr ? a.a_rows[m0 + r] : r) * a.lda);
}
__device__ __forceinline__ unsigned w_offset(const Tile& a, int n0, int j) {
  if (a.epi.kind < EPI_GATE) return (unsigned)(min(j, a.N - 1 - n0) * a.ldw);
  const int half = a.N >> 1;
  return (unsigned)((min((j >> 5) * 16 + (j & 15), half - 1 - (n0 >> 1)) + ((j >> 4) & 1) * half) * a.ldw);
}
__device__ __forceinline__ const char* a_base(const Tile& a, const char* A, int m0) { return a.a_rows != nullptr ? A : A + (size_t)m0 * a.lda; }
__device__ __forceinline__ const char* w_base(const Tile& a, const char* W, int n0) {
  return W + (size_t)(a.epi.kind < EPI_GATE ? n0 : n0 >> 1) * a.ldw;
}

// (offsets of a tile stay below 2^31: the host checks)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* base, bool live) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, live ? 0x7fffffff : 0, 0x00020000);
}

// four consecutive columns as fp32, or rounded to nearest even as bf16
template <int TC>
__device__ __forceinline__ void store4(void* C, size_t idx, floatx4 v) {
  if constexpr (TC == 1) {
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16_t*>(C) + idx) = __builtin_convertvector(v, bf16x4);
  } else {
    *reinterpret_cast<floatx4*>(reinterpret_cast<float*>(C) + idx) = v;
  }
}

// (ACC: the accumulators are in accumulation registers, written by asm; each stays there until it is used)
template <bool ACC>
__device__ __forceinline__ void hold(floatx4& c) {
  if constexpr (ACC) asm volatile("" : "+a"(c));
}

// A wave's outputs: acc[u][t] = rows mw + 16 u + (lane & 15), columns nw + 16 t + 4 (lane >> 4) .. + 3.  The wave lays them down in its
// own piece of LDS (PU row groups at a time) and takes them up row by row, so that a store covers whole rows of the tile (straight from the
// registers it was pieces of 32 or 64 bytes of 16 rows: 16384 x 4096 x 4096 404 -> 392 us, 9692 x 10880 x 2048 390 -> 340) and an
// activation is a short loop: unrolled over all accumulators its code would be larger than the cache.
template <int NJ, bool ACC>
__device__ __forceinline__ void lay_down(floatx4 (&row)[NJ], int u, char* lds) {
  constexpr int CH = 4 * NJ;
  const int lane = threadIdx.x & 63, fr = lane & 15, grp = lane >> 4, r = u * 16 + fr;
#pragma unroll
  for (int t = 0; t < NJ; ++t) {
    hold<ACC>(row[t]);
    *reinterpret_cast<floatx4*>(lds + (r * CH + ((4 * t + grp) ^ (r & (CH - 1)))) * 16) = row[t];
  }
}

// The rows that a wave laid down: a loop for each kind of epilogue.  With the kind asked for at each value the loop was a chain of
// branches over the other kinds' code, and a wave that has its SIMD to itself waits for the instructions after each: 16384 x 14336 x
// 4096 with xIELU 1827 us, 1523 so (branches in xIELU itself: 1572); 9692 x 10880 x 2048 silu gates 469 and 362.
template <int NJ, int TC, int KIND>
__device__ __forceinline__ void value_rows(const Tile& a, const EpiRegs (&er)[4], floatx4 b, size_t cbase, int m0, int rows, int n, int mend, const char* lds) {
  constexpr int CH = 4 * NJ, RI = 64 / CH;          // 16-byte chunks of a row; rows per step of the loop
  const int lane = threadIdx.x & 63, c = lane % CH;
#pragma unroll 2
  for (int i = 0; i < rows; i += RI) {
    const int r = i + lane / CH;
    floatx4 v = *reinterpret_cast<const floatx4*>(lds + (r * CH + (c ^ (r & (CH - 1)))) * 16) + b;
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = epi_value_of<KIND>(v[x], a.epi, er[x]);
    if (m0 + r < mend && n < a.N) store4<TC>(a.C, cbase + (size_t)(m0 + r) * a.ldc + n, v);
  }
}
template <int NJ, int TC, int KIND>
__device__ __forceinline__ void gate_rows(const Tile& a, int m0, int rows, int nw, int mend, const char* lds) {
  constexpr int CH = 4 * NJ, RI = 64 / CH;
  const int lane = threadIdx.x & 63, c = lane % (CH / 2), cg = (c >> 2) * 8 + (c & 3);      // column chunk, its gate chunk (the up chunk: + 4)
  const int n = (nw >> 1) + 4 * c;
#pragma unroll 2
  for (int i = 0; i < rows; i += 2 * RI) {
    const int r = i + lane / (CH / 2);
    const floatx4 g = *reinterpret_cast<const floatx4*>(lds + (r * CH + (cg ^ (r & (CH - 1)))) * 16);
    const floatx4 u = *reinterpret_cast<const floatx4*>(lds + (r * CH + ((cg + 4) ^ (r & (CH - 1)))) * 16);
    floatx4 v;
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = epi_gate_of<KIND>(g[x], u[x], a.epi);
    if (m0 + r < mend && n < (a.N >> 1)) store4<TC>(a.C, (size_t)(m0 + r) * a.ldc + n, v);
  }
}

// One pass: the wave's rows m0 .. m0 + rows - 1, which it has laid down.
template <int NJ, int TC>
__device__ __forceinline__ void rows_out(const Tile& a, const EpiRegs (&er)[4], floatx4 b, size_t cbase, int m0, int rows, int nw, int mend, const char* lds) {
  const Epi& e = a.epi;
  const int n = nw + 4 * ((int)(threadIdx.x & 63) % (4 * NJ));
  if (NJ >= 2 && e.kind >= EPI_GATE) {               // (no bias: the gated products have none)
    if (e.kind == EPI_GATE) gate_rows<NJ, TC, EPI_GATE>(a, m0, rows, nw, mend, lds);
    else if (e.kind == EPI_GATE + 1) gate_rows<NJ, TC, EPI_GATE + 1>(a, m0, rows, nw, mend, lds);
    else gate_rows<NJ, TC, EPI_GATE + 2>(a, m0, rows, nw, mend, lds);
    return;
  }
  switch (e.kind) {
    case EPI_XIELU: value_rows<NJ, TC, EPI_XIELU>(a, er, b, cbase, m0, rows, n, mend, lds); break;
    case EPI_RELU2: value_rows<NJ, TC, EPI_RELU2>(a, er, b, cbase, m0, rows, n, mend, lds); break;
    case EPI_DECAY: value_rows<NJ, TC, EPI_DECAY>(a, er, b, cbase, m0, rows, n, mend, lds); break;
    case EPI_SOFTCAP: value_rows<NJ, TC, EPI_SOFTCAP>(a, er, b, cbase, m0, rows, n, mend, lds); break;
    case EPI_SCALE: value_rows<NJ, TC, EPI_SCALE>(a, er, b, cbase, m0, rows, n, mend, lds); break;
    default: value_rows<NJ, TC, 0>(a, er, b, cbase, m0, rows, n, mend, lds);
  }
}
// What a wave's columns need besides (lane: four columns from n on).
__device__ __forceinline__ floatx4 column_terms(const Tile& a, EpiRegs (&er)[4], size_t cbase, int n) {
  const Epi& e = a.epi;
  const EpiRegs er0 = epi_regs(e);
  floatx4 b = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; ++i) er[i] = er0;
  if (e.kind < EPI_GATE && n < a.N) {
#pragma unroll
    for (int i = 0; i < 4; ++i) epi_column(e, er[i], n + i);
    if (e.bias != nullptr) b = *reinterpret_cast<const floatx4*>(e.bias + cbase + n);
  }
  return b;
}

template <int MI, int NJ, int TC>
__device__ __forceinline__ void finish_as(const Tile& a, floatx4 (&acc)[MI][NJ], size_t cbase, int mw, int nw, int mend, char* lds) {
  const int lane = threadIdx.x & 63, fr = lane & 15, grp = lane >> 4;
  if (a.ragged) {                                           // (plain products of few columns: a column at a time)
#pragma unroll
    for (int t = 0; t < NJ; ++t)
#pragma unroll
      for (int u = 0; u < MI; ++u)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int n = nw + t * 16 + 4 * grp + x, m = mw + u * 16 + fr;
          const size_t at = cbase + (size_t)m * a.ldc + n;
          if (n >= a.N || m >= mend) continue;
          if constexpr (TC == 1) reinterpret_cast<bf16_t*>(a.C)[at] = f_to_bf16(acc[u][t][x]);
          else reinterpret_cast<float*>(a.C)[at] = acc[u][t][x];
        }
    return;
  }
  EpiRegs er[4];
  const floatx4 b = column_terms(a, er, cbase, nw + 4 * (lane % (4 * NJ)));
#pragma unroll
  for (int u = 0; u < MI; ++u) lay_down<NJ, false>(acc[u], u, lds);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // (the wave's own rows: no other wave reads them)
  rows_out<NJ, TC>(a, er, b, cbase, mw, 16 * MI, nw, mend, lds);
}
template <int MI, int NJ>
__device__ __forceinline__ void finish(const Tile& a, floatx4 (&acc)[MI][NJ], size_t cbase, int mw, int nw, int mend, char* lds) {
  if (a.epi.tc == 1) finish_as<MI, NJ, 1>(a, acc, cbase, mw, nw, mend, lds);
  else finish_as<MI, NJ, 0>(a, acc, cbase, mw, nw, mend, lds);
}

// The same for the large tiles' U x 8 accumulators, PU row groups a pass; those past the eighth group are in vector registers.
template <int U, int PU, int TC, int P = 0>
__device__ __forceinline__ void finish_big(const Tile& a, floatx4 (&acc)[U < 8 ? U : 8][8], floatx4 (&more)[U > 8 ? U - 8 : 1][8], const EpiRegs (&er)[4],
                                           floatx4 b, size_t cbase, int mw, int nw, int mend, char* lds) {
  constexpr int N = U - P < PU ? U - P : PU;
#pragma unroll
  for (int u = 0; u < N; ++u) {
    if (P + u < 8) lay_down<8, true>(acc[P + u < 8 ? P + u : 0], u, lds);
    else lay_down<8, false>(more[P + u < 8 ? 0 : P + u - 8], u, lds);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  rows_out<8, TC>(a, er, b, cbase, mw + 16 * P, 16 * N, nw, mend, lds);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if constexpr (P + PU < U) finish_big<U, PU, TC, P + PU>(a, acc, more, er, b, cbase, mw, nw, mend, lds);
}

// ------------------------------------------------------------------------------------ 32 U x 256: 128, 160 .. 320 rows
// Four waves, one per SIMD, 16 U x 128 outputs each.  U = 8: 128 x 128, all 256 accumulation registers of a wave, a fragment
// read from LDS feeds 8 MFMAs; U = 9 and 10 hold their last row groups in vector registers and all of LDS.  Heights other than 256 are for row
// counts that leave the chip idle in the last (or only) round of 256-row tiles: 8536 x 2048 x 2048 takes 272 tiles of 256 rows, 77 us, and 240
// of 288 rows, 60 us (320: 65, 160: 72); x 5440 192 rows 178, 288 147; 6722 x 2048 x 2048 192 rows 54, 224 50 - 53.  Over 500 random long
// products of up to 20,000 rows the four heights beside 128, 192 and 256 give 3% on average.
// The products are written as in-place asm so that the accumulators stay where they are (with no spare accumulation register the
// compiler would otherwise copy them) and so that LDS reads and DMAs keep their places between them; reads run one phase of 8 MFMAs
// a row group ahead, DMAs three half-tiles, one barrier per two phases.
namespace t256 {
constexpr int TN = 256, KT = 128 /* bytes of a K tile's row */;
constexpr int lds_bytes(int u) { return 2 * (32 * u + TN) * KT; }
}

template <bool ACC>
__device__ __forceinline__ void mfma_in_place(floatx4& c, const bf16x8& a, const bf16x8& b) {
  if constexpr (ACC) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b) : "memory");
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b) : "memory");
}

// U: 16-row groups of a wave; they are taken in two halves, the first of H0, the second of U - H0.
template <int U>
__device__ __forceinline__ void tile_256(const Tile& a) {
  using namespace t256;
  constexpr int H0 = (U + 1) / 2, H1 = U / 2, TM = 32 * U, WIMG = TM * KT, STG = WIMG + TN * KT;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const char *A, *W;
  size_t cbase;
  int m0, mend, n0;
  if (!locate<TM, TN>(a, A, W, cbase, m0, mend, n0)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // DMA: a half-tile is 16 pieces (A: 4 H0 or 4 H1) of eight rows, half of them for either half of the waves: piece j of W is rows
  // (j >> 3) 128 + (j & 7) 8 (+ 64: the second half); a wave moves pieces 4 wave .. + 3 (A: H0 or H1)
  const int lr = lane >> 3, lc = (lane & 7) ^ lr;
  int xpr[2][H0], wpr[4];
  unsigned xo[2][H0], wo[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = 4 * wave + i;
    wpr[i] = (j >> 3) * 128 + (j & 7) * 8;
#pragma unroll
    for (int h = 0; h < 2; ++h) wo[4 * h + i] = w_offset(a, n0, wpr[i] + 64 * h + lr) + lc * 16;
  }
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < (h ? H1 : H0); ++i) {
      const int n = h ? H1 : H0, j = n * wave + i;
      xpr[h][i] = j / (2 * n) * (16 * U) + h * 16 * H0 + j % (2 * n) * 8;
      xo[h][i] = a_offset(a, m0, mend, xpr[h][i] + lr) + lc * 16;
    }
  const char* Ab = a_base(a, A, m0);
  const char* Wb = w_base(a, W, n0);
  // (past the last K tile the DMAs go through a descriptor of no records: counted like the others, they write zeros)
  const __amdgpu_buffer_rsrc_t rA = rsrc_of(Ab, true), rW = rsrc_of(Wb, true), r0 = rsrc_of(Ab, false);
#define T_DMA(rs, off, k0, dst) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LDS_AS void*)(dst), 16, off, k0, 0, 0)
#define T_X(rs, buf, h, i, k0) T_DMA(rs, xo[h][i], k0, smem + (buf) * STG + xpr[h][i] * 128)
#define T_W(rs, buf, h, i, k0) T_DMA(rs, wo[(h) * 4 + (i)], k0, smem + (buf) * STG + WIMG + (wpr[i] + (h) * 64) * 128)
  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane & 15, grp = lane >> 4, sw = fr & 7;
  const int c0 = (grp ^ sw) << 4, c1 = ((4 + grp) ^ sw) << 4;
  const int xrow = (wm * 16 * U + fr) * 128, wrow = WIMG + (wn * 128 + fr) * 128;
  floatx4 acc[U < 8 ? U : 8][8], more[U > 8 ? U - 8 : 1][8];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int t = 0; t < 8; ++t) (u < 8 ? acc[u < 8 ? u : 0] : more[u < 8 ? 0 : u - 8])[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16x8 xf[U][2], wf[8][2];
#define T_HOLD()                                                                                   \
  _Pragma("unroll") for (int u_ = 0; u_ < (U < 8 ? U : 8); ++u_)                                   \
  _Pragma("unroll") for (int t_ = 0; t_ < 8; ++t_) asm volatile("" : "+a"(acc[u_][t_]));           \
  _Pragma("unroll") for (int u_ = 8; u_ < U; ++u_)                                                 \
  _Pragma("unroll") for (int t_ = 0; t_ < 8; ++t_) asm volatile("" : "+v"(more[u_ < 8 ? 0 : u_ - 8][t_]));
  T_HOLD();
  asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");          // (the zeros are written before the first MFMA reads them)
#define T_RX(buf, f, k) xf[f][k] = *(const bf16x8*)(smem + (buf) * STG + xrow + (f) * 2048 + ((k) ? c1 : c0))
#define T_RW(buf, f, k) wf[f][k] = *(const bf16x8*)(smem + (buf) * STG + wrow + (f) * 2048 + ((k) ? c1 : c0))
// 8 MFMAs a row group of the quadrant (x half xh, w half wh); after the first even ones the reads of the half needed next (RX: of x), two a row
// group or 8 of them, after later ones the DMAs of a half-tile (DX: of x)
#define T_PHASE(xh, wh, RX, rbuf, rh, DX, rs, dbuf, dh, dk, SYNC)                                  \
  {                                                                                                \
    constexpr int HN_ = (xh) ? H1 : H0, RN_ = (rh) ? H1 : H0, DN_ = DX ? ((dh) ? H1 : H0) : 4;     \
    constexpr int D0_ = HN_ == 5 ? 25 : HN_ == 4 ? 17 : HN_ == 3 ? 13 : 5;                         \
    _Pragma("unroll") for (int i_ = 0; i_ < 8 * HN_; ++i_) {                                       \
      const int s_ = i_ / (4 * HN_), u_ = (xh) * H0 + (i_ >> 2) % HN_, t_ = (wh) * 4 + (i_ & 3);   \
      if (u_ < 8) mfma_in_place<true>(acc[u_ < 8 ? u_ : 0][t_], wf[t_][s_], xf[u_][s_]);           \
      else mfma_in_place<false>(more[u_ < 8 ? 0 : u_ - 8][t_], wf[t_][s_], xf[u_][s_]);            \
      if (i_ < (RX ? 4 * RN_ : 16) && (i_ & 1) == 0) {                                             \
        const int f_ = i_ >> 2, k_ = (i_ >> 1) & 1;                                                \
        if (RX) T_RX(rbuf, (rh) * H0 + f_, k_);                                                    \
        else T_RW(rbuf, (rh) * 4 + f_, k_);                                                        \
      }                                                                                            \
      if (i_ >= D0_ && i_ < D0_ + 3 * DN_ && (i_ - D0_) % 3 == 0) {                                \
        if (DX) T_X(rs, dbuf, dh, (i_ - D0_) / 3, dk);                                             \
        else T_W(rs, dbuf, dh, (i_ - D0_) / 3, dk);                                                \
      }                                                                                            \
    }                                                                                              \
    if (SYNC) {                                                                                    \
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(U + 8) : "memory");                      \
      __builtin_amdgcn_s_barrier();                                                                \
    }                                                                                              \
  }
// a K tile held by buffer 0: w halves 0, 1; by buffer 1: w halves 1, 0 (each phase reads one half for the next one)
#define T_EVEN(rx, rw, dk)                                                                         \
  T_PHASE(0, 0, 0, 0, 1, 1, rx, 0, 0, dk, 0)                                                       \
  T_PHASE(0, 1, 1, 0, 1, 0, rw, 0, 0, dk, 1)                                                       \
  T_PHASE(1, 1, 1, 1, 0, 0, rw, 0, 1, dk, 0)                                                       \
  T_PHASE(1, 0, 0, 1, 1, 1, rx, 0, 1, dk, 1)
#define T_ODD(rx, rw, dk)                                                                          \
  T_PHASE(0, 1, 0, 1, 0, 1, rx, 1, 0, dk, 0)                                                       \
  T_PHASE(0, 0, 1, 1, 1, 0, rw, 1, 1, dk, 1)                                                       \
  T_PHASE(1, 0, 1, 0, 0, 0, rw, 1, 0, dk, 0)                                                       \
  T_PHASE(1, 1, 0, 0, 0, 1, rx, 1, 1, dk, 1)
  const int nk = a.nk;
  {
    const __amdgpu_buffer_rsrc_t rA1 = nk > 1 ? rA : r0, rW1 = nk > 1 ? rW : r0;
    const int k1 = nk > 1 ? KT : 0;
#pragma unroll
    for (int i = 0; i < H0; ++i) T_X(rA, 0, 0, i, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) T_W(rW, 0, 0, i, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) T_W(rW, 0, 1, i, 0);
#pragma unroll
    for (int i = 0; i < H1; ++i) T_X(rA, 0, 1, i, 0);
#pragma unroll
    for (int i = 0; i < H0; ++i) T_X(rA1, 1, 0, i, k1);
#pragma unroll
    for (int i = 0; i < 4; ++i) T_W(rW1, 1, 1, i, k1);
#pragma unroll
    for (int i = 0; i < 4; ++i) T_W(rW1, 1, 0, i, k1);
#pragma unroll
    for (int i = 0; i < H1; ++i) T_X(rA1, 1, 1, i, k1);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(U + H1 + 12) : "memory");
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int f = 0; f < H0 || f < 4; ++f) {
    if (f < H0) { T_RX(0, f, 0); T_RX(0, f, 1); }
    if (f < 4) { T_RW(0, f, 0); T_RW(0, f, 1); }
  }
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(U + 8) : "memory");
  __builtin_amdgcn_s_barrier();
  // (an odd last K tile is followed by one of zeros, which is what a DMA without records leaves in LDS: a loop exit in the
  // middle would have the compiler move accumulators between registers while asm MFMAs it cannot see are still writing them)
  int kt = 0;
  do {
    const bool more2 = kt + 2 < nk, more3 = kt + 3 < nk;
    const int k2 = more2 ? (kt + 2) * KT : 0, k3 = more3 ? (kt + 3) * KT : 0;
    const __amdgpu_buffer_rsrc_t rx2 = more2 ? rA : r0, rw2 = more2 ? rW : r0, rx3 = more3 ? rA : r0, rw3 = more3 ? rW : r0;
    T_EVEN(rx2, rw2, k2)
    T_ODD(rx3, rw3, k3)
    asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");      // (the last MFMAs' passes, before anything may move an accumulator)
    kt += 2;
  } while (kt < nk);
  // every DMA has landed and every wave is done with the tiles before LDS changes its use; the nops give the last MFMAs,
  // which the compiler cannot see, their passes before the accumulators are read
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#undef T_HOLD
#undef T_RX
#undef T_RW
#undef T_PHASE
#undef T_EVEN
#undef T_ODD
#undef T_X
#undef T_W
  constexpr int FIT = 2 * STG / (4 * 8192), PASSES = (U + FIT - 1) / FIT, PU = (U + PASSES - 1) / PASSES;      // row groups that a wave's share of LDS holds
  char* const mine = smem + wave * (PU * 8192);
  const int mw = m0 + wm * 16 * U, nw = n0 + wn * 128;
  EpiRegs er[4];
  const floatx4 b = column_terms(a, er, cbase, nw + 4 * (lane % 32));
  if (a.epi.tc == 1) finish_big<U, PU, 1>(a, acc, more, er, b, cbase, mw, nw, mend, mine);
  else finish_big<U, PU, 0>(a, acc, more, er, b, cbase, mw, nw, mend, mine);
}

template <int U>
__global__ __launch_bounds__(256, 1) void gemm_tile_big(Tile a) { tile_256<U>(a); }

// ------------------------------------------------------------------------------------ smaller tiles
// 32 MI x 32 NJ outputs, four waves in a 2 x 2 grid of 16 MI x 16 NJ, S stages of LDS: the DMAs of K tile t + S - 1 are issued
// while tile t is multiplied, one barrier per K tile.  What bounds them is the chain of one K tile (wait, barrier, LDS read,
// MFMA), 0.5 us or more for one wave a SIMD whatever the tile: KG groups of four waves take every KG-th K tile each, so that a
// SIMD has KG chains to run (256 x 2048 x 2048 in 64 x 64 tiles: 16 us with one group, 12 with two).
//
// A K tile is a 128-byte row of W: 64 bf16 (two 16x16x32 MFMAs per fragment pair) or 32 fp32 (eight 16x16x4 MFMAs: lane group g
// holds elements 4 g .. 4 g + 3 of 16, and MFMA i multiplies the i-th ones).  fp32 rows against bf16 weights come in as they
// are, 256 bytes a row, and are rounded when a fragment is read.
template <typename T> struct Frag;
template <> struct Frag<bf16_t> { typedef bf16x8 V; };
template <> struct Frag<float> { typedef floatx4 V; };
__device__ __forceinline__ floatx4 mfma_frag(const bf16x8& w, const bf16x8& x, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, c, 0, 0, 0);
}
__device__ __forceinline__ floatx4 mfma_frag(const floatx4& w, const floatx4& x, floatx4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], c, 0, 0, 0);
  return c;
}

// (even and odd terms of four in sums of their own)
__device__ __forceinline__ void mfma_frag(const floatx4& w, const floatx4& x, floatx4& c, floatx4& odd) {
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], c, 0, 0, 0);
    odd = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i + 1], x[i + 1], odd, 0, 0, 0);
  }
}

// the DMAs of K tile kt: PX pieces of A (128 XS bytes a row), PW of W
template <int PX, int PW, int XS, int XIMG>
__device__ __forceinline__ void fill(const char* Ab, const char* Wb, int kt, int nk, int wave, const unsigned* xo, const unsigned* wo, char* stg) {
  const bool live = kt < nk;             // (past the last K tile: a descriptor of no records, counted like the others; it leaves zeros)
  const __amdgpu_buffer_rsrc_t ra = rsrc_of(Ab, live), rw = rsrc_of(Wb, live);
  const int k0 = live ? kt * 128 : 0;
#pragma unroll
  for (int i = 0; i < PX; ++i) T_DMA(ra, xo[i], k0 * XS, stg + (PX * wave + i) * 1024);
#pragma unroll
  for (int i = 0; i < PW; ++i) T_DMA(rw, wo[i], k0, stg + XIMG + (PW * wave + i) * 1024);
}

template <typename TA, typename TW, int MI, int NJ, int S, int OCC, int KG>
__global__ __launch_bounds__(256 * KG, OCC * KG) void gemm_tile_mid(Tile a) {
  typedef typename Frag<TW>::V V;
  constexpr int XS = sizeof(TA) / sizeof(TW);               // 2: fp32 rows against bf16 weights
  constexpr int TM = 32 * MI, TN = 32 * NJ, XIMG = TM * 128 * XS, STG = XIMG + TN * 128, PX = MI * XS, PW = NJ;
  extern __shared__ __attribute__((aligned(16))) char smem_all[];
  const char *A, *W;
  size_t cbase;
  int m0, mend, n0;
  if (!locate<TM, TN>(a, A, W, cbase, m0, mend, n0)) return;
  const int lane = threadIdx.x & 63;
  const int wall = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wall & 3, kg = wall >> 2;
  char* smem = smem_all + kg * (S * STG);
  const int lr = lane >> 3, lc = (lane & 7) ^ lr;
  unsigned xo[PX], wo[PW];
#pragma unroll
  for (int i = 0; i < PX; ++i) {
    if constexpr (XS == 1) {
      xo[i] = a_offset(a, m0, mend, (PX * wave + i) * 8 + lr) + lc * 16;
    } else {                                                 // pieces of 4 rows x 256 bytes, chunk c of row r in slot c ^ (r & 15)
      const int r = (PX * wave + i) * 4 + (lane >> 4);
      xo[i] = a_offset(a, m0, mend, r) + ((lane ^ r) & 15) * 16;
    }
  }
#pragma unroll
  for (int i = 0; i < PW; ++i) wo[i] = w_offset(a, n0, (PW * wave + i) * 8 + lr) + lc * 16;
  const char* Ab = uniform(a_base(a, A, m0));
  const char* Wb = uniform(w_base(a, W, n0));
  const int nk = a.nk;
  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane & 15, grp = lane >> 4, sw = fr & 7;
  const int c0 = (grp ^ sw) << 4, c1 = ((4 + grp) ^ sw) << 4;
  const int xrow = (wm * 16 * MI + fr) * 128 * XS, wrow = XIMG + (wn * 16 * NJ + fr) * 128;
  // (small tiles of one wave group: sums of a part of the terms each, as several groups have them.  One of all in a row is further from 64
  // bits: fp32, 2048 terms 8.1e-7, 5.8e-7 in two sums and 4.1e-7 in four, for the same time)
  constexpr int SUMS = KG > 1 || MI * NJ > 8 ? 1 : sizeof(TW) == 4 && MI * NJ <= 4 ? 4 : 2;
  floatx4 sums[SUMS][MI][NJ], (&acc)[MI][NJ] = sums[0];
#pragma unroll
  for (int i = 0; i < SUMS; ++i)
#pragma unroll
    for (int u = 0; u < MI; ++u)
#pragma unroll
      for (int t = 0; t < NJ; ++t) sums[i][u][t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < S - 1; ++s) fill<PX, PW, XS, XIMG>(Ab, Wb, s * KG + kg, nk, wave, xo, wo, smem + s * STG);
  int cur = 0, nxt = S - 1;
  for (int kt = kg; kt < nk + kg; kt += KG) {               // (every group as often as the first: they share the barriers)
    // this wave's pieces of tile kt have landed and its reads of the tile before are done; after the barrier, everyone's
    asm volatile("" ::: "memory");
    constexpr int LEFT = (S - 2) * (PX + PW);               // DMAs of later K tiles that may stay in flight
    __builtin_amdgcn_s_waitcnt((LEFT & 15) | (LEFT >> 4) << 14 | 0x70);       // vmcnt(LEFT) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fill<PX, PW, XS, XIMG>(Ab, Wb, kt + (S - 1) * KG, nk, wave, xo, wo, smem + nxt * STG);
    const char* stg = smem + cur * STG;
    V x[2][MI], w[2][NJ];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int c = k ? c1 : c0;
#pragma unroll
      for (int u = 0; u < MI; ++u) {
        if constexpr (XS == 1) {
          x[k][u] = *(const V*)(stg + xrow + u * 2048 + c);
        } else {
          typedef float floatx8 __attribute__((ext_vector_type(8)));
          const char* row = stg + xrow + u * 4096;
          const floatx4 lo = *(const floatx4*)(row + (((8 * k + 2 * grp) ^ fr) << 4)), hi = *(const floatx4*)(row + (((8 * k + 2 * grp + 1) ^ fr) << 4));
          x[k][u] = __builtin_convertvector((floatx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}), V);
        }
      }
#pragma unroll
      for (int t = 0; t < NJ; ++t) w[k][t] = *(const V*)(stg + wrow + t * 2048 + c);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int u = 0; u < MI; ++u)
#pragma unroll
        for (int t = 0; t < NJ; ++t) {
          if constexpr (SUMS == 4) mfma_frag(w[k][t], x[k][u], sums[2 * k][u][t], sums[2 * k + 1][u][t]);
          else sums[k % SUMS][u][t] = mfma_frag(w[k][t], x[k][u], sums[k % SUMS][u][t]);
        }
    cur = cur + 1 == S ? 0 : cur + 1;
    nxt = nxt + 1 == S ? 0 : nxt + 1;
  }
#pragma unroll
  for (int u = 0; u < MI; ++u)
#pragma unroll
    for (int t = 0; t < NJ; ++t) {
      if constexpr (SUMS == 4) acc[u][t] = (acc[u][t] + sums[SUMS - 3][u][t]) + (sums[SUMS - 2][u][t] + sums[SUMS - 1][u][t]);
      else if constexpr (SUMS == 2) acc[u][t] += sums[1][u][t];
    }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  constexpr int OUT = 16 * MI * 16 * NJ * 4;                // a wave's accumulators
  static_assert(4 * OUT * (KG > 1 ? KG - 1 : 1) <= KG * S * STG, "the accumulators fit the stages");
  if constexpr (KG > 1) {                                    // the wave groups' partial sums meet in LDS, in the groups' order
    if (kg > 0) {
#pragma unroll
      for (int u = 0; u < MI; ++u)
#pragma unroll
        for (int t = 0; t < NJ; ++t)
          *reinterpret_cast<floatx4*>(smem_all + ((kg - 1) * 4 + wave) * OUT + ((u * NJ + t) * 64 + lane) * 16) = acc[u][t];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int g = 1; g < KG; ++g)
#pragma unroll
      for (int u = 0; u < MI; ++u)
#pragma unroll
        for (int t = 0; t < NJ; ++t)
          acc[u][t] += *reinterpret_cast<const floatx4*>(smem_all + ((g - 1) * 4 + wave) * OUT + ((u * NJ + t) * 64 + lane) * 16);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // (the same wave lays its rows down in the same place)
  }
  finish<MI, NJ>(a, acc, cbase, m0 + wm * 16 * MI, n0 + wn * 16 * NJ, mend, smem_all + wave * OUT);
}
#undef T_DMA

int pick_order(int tiles_m, int tiles_n) {
  if (tiles_n % 8 == 0)
    for (int g = 4; g <= 8; ++g)
      if ((tiles_n / 8) % g == 0) return -g;
  if (tiles_m % 8 == 0)
    for (int g = 4; g <= 8; ++g)
      if ((tiles_m / 8) % g == 0) return g;
  return -4;
}

template <auto KERNEL>
int start(int tm, int tn, int threads, int lds, Tile t, hipStream_t s) {
  // (row groups: each may end in a tile of its own)
  t.tiles_m = (t.M + tm - 1) / tm + (t.offs != nullptr ? t.groups - 1 : 0);
  t.tiles_n = (t.N + tn - 1) / tn;
  t.order = pick_order(t.tiles_m, t.tiles_n);
  static const hipError_t e = hipFuncSetAttribute((const void*)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return -(int)e;
  hipLaunchKernelGGL(KERNEL, dim3(t.tiles_m * t.tiles_n, t.offs == nullptr ? t.groups : 1), dim3(threads), lds, s, t);
  const hipError_t l = hipGetLastError();
  return l == hipSuccess ? 1 : -(int)l;
}

}  // namespace

// The tiles, and what a launch of each costs: rounds of `slots` blocks (what the chip holds at once), each nk K tiles and
// a start and a store.  A launch that leaves CUs idle in its last (or only) round wants smaller tiles, a long one the large tile; the
// cheapest sum wins.  us per K tile and per round for products of few K tiles, measured on full rounds at K = 128 .. 8192, and for those of
// at least LONG (least squares of the relative error over 400, 120 and 100 random products of 64 .. 20,000 rows with cold weights), where a round
// that fills a part of the chip takes PART of a full one's time a K tile and more by its share (the clock rises).  The second kind of
// product takes 1.009 of the best tile's time on average (1.026 by the first figures); below LONG they are no better than the first.  Row groups
// stay with the first: their sizes and the blocks' share of a cold W decide, and of 400 random ones 31 were more than 4% slower by the
// second (and 1% faster on average).
struct TileCost { int tm, tn, slots; float k_us, round_us, k_long, round_long; bool shared = false; };      // shared: only where a CU gets several blocks
static const int LONG = 18;
static const float PART = 0.8f;
// bf16 (16384 x 14336 x 4096: the 256 tile 1.49 ms, 128 x 128 2.05; 1024 x 2048 x 2048: 64 x 128 14 us, the 256 tile 42;
// 256 x 2048 x 2048: 32 x 64 8 us, the 256 tile 41)
static const TileCost TILES[] = {{256, 256, 256, 1.42f, 11.f, 1.263f, 11.816f},     // least LDS and L2 traffic per product: 1.24 - 1.45 PFLOP/s at 16384 rows
                                 {128, 128, 512, 1.08f, 5.f, 0.818f, 5.367f},       // two blocks a CU
                                 {128, 128, 256, 0.55f, 6.f, 0.552f, 5.788f}, {64, 128, 256, 0.40f, 5.f, 0.315f, 4.453f},      // two wave groups
                                 {64, 64, 256, 0.26f, 3.f, 0.2f, 3.425f},
                                 {32, 64, 256, 0.16f, 3.5f, 0.137f, 3.665f}, {32, 32, 256, 0.12f, 3.5f, 0.089f, 3.092f},       // four
                                 {192, 256, 256, 1.09f, 9.5f, 0.945f, 9.866f}, {128, 256, 256, 0.82f, 8.f, 0.733f, 7.441f},
                                 // long products only: two blocks a CU, which stand at barriers of their own (1024 x 4096 x 2048 23.6 us, 24.6 on
                                 // 128 x 128, 28.2 on two wave groups), and the heights between and above those of 256 columns (above: 8536 x 2048 x
                                 // 2048), at 1.02 of what was fitted: products of many rounds are within 2% of each other on tiles of 256 rows and more, and bound by power
                                 {64, 128, 512, 0.f, 0.f, 0.455f, 4.821f}, {160, 256, 256, 0.f, 0.f, 0.876f, 8.85f}, {224, 256, 256, 0.f, 0.f, 1.112f, 11.8f},
                                 {288, 256, 256, 0.f, 0.f, 1.362f, 14.47f}, {320, 256, 256, 0.f, 0.f, 1.488f, 15.77f}};
// fp32 rows, bf16 weights.  64 x 128 on two blocks a CU with two stages each, whose loads, products and stores run beside one another's (before, 128 x 128
// on one block with three: 2048 x 2048 x 2048 38 us, so 29; 8192 rows 141, 114; 9692 x 2048 x 128 35, 25; 16384 rows of 16 blocks x 256, two sets of weights 384, 321)
static const TileCost TILES_MIXED[] = {{64, 128, 512, 0.66f, 4.5f, 0.66f, 7.2f}, {64, 128, 256, 0.47f, 5.f, 0.561f, 3.771f}, {64, 64, 256, 0.37f, 4.2f, 0.313f, 3.17f},
                                       {64, 64, 512, 0.6f, 4.f, 0.476f, 3.454f},    // two blocks a CU
                                       {32, 32, 256, 0.16f, 3.5f, 0.137f, 3.025f}};
// fp32 (bound by the fp32 MFMA's 150 TFLOP/s; 400 x 2048 x 8192: 64 x 64 165 us, 128 x 128 573; 1000 x 2048 x 2048: 64 x 128 71 us,
// 128 x 128 129)
static const TileCost TILES_F32[] = {{128, 128, 512, 4.0f, 8.f, 3.7f, 8.f}, {128, 128, 256, 2.15f, 6.f, 1.934f, 6.092f}, {64, 128, 256, 1.1f, 6.f, 1.05f, 4.441f},
                                     {64, 64, 256, 0.63f, 4.f, 0.573f, 3.127f}, {32, 64, 256, 0.33f, 4.f, 0.294f, 3.226f}, {32, 32, 256, 0.195f, 4.f, 0.166f, 2.685f},
                                     // long products only: three blocks a CU keep its matrix units busy between them, so that a round is of 256 (1200 x 8192 x
                                     // 2048 306 us, 343 on 64 x 128; x 4384 185, 205; x 2048 95, 101; one block a CU alone is slower: 400 x 2048 x 8192 156, 143;
                                     // row groups above five rounds, as their sizes fall: 150 random ones 0.95 of the time)
                                     {64, 64, 256, 0.f, 0.f, 0.475f, 0.5f, true}};

static int pick_tile(const TileCost* tiles, int count, float part, int M, int N, int nk, int groups, bool by_rows, bool gated) {
  int best = -1;
  float least = 0.f;
  for (int v = 0; v < count; ++v) {
    const TileCost& t = tiles[v];
    const bool lng = nk >= LONG && (!by_rows || t.shared);
    if ((gated && t.tn < 64) || (t.k_us == 0.f && !lng)) continue;      // (a wave of the 32-column tile has one half of a gated column only)
    const float k = (float)nk * (lng ? t.k_long : t.k_us), round = lng ? t.round_long : t.round_us;
    // (row groups: their sizes are on the device; each ends in a part of a tile, half of one on average, and how they fall on the
    // CUs is chance: a launch that just fills the chip takes a second round, 2048 rows of 8 experts on 192-row tiles 80 us, 62 on 256)
    const long long cols = (N + t.tn - 1) / t.tn;
    float us;
    if (by_rows) {
      const float full = ((float)M / t.tm + 0.5f * groups) * cols / t.slots;
      if (t.shared && full <= 5.f) continue;
      us = (full <= 0.9f ? 1.f : full + 0.5f) * (k + round);
    } else {
      const long long blocks = (long long)((M + t.tm - 1) / t.tm) * groups * cols, rest = blocks % t.slots;
      if (t.shared && blocks <= t.slots) continue;
      us = (float)(blocks / t.slots) * (k + round);
      if (rest) us += k * (lng ? part + (1.f - part) * (float)rest / t.slots : 1.f) + round;
    }
    if (best < 0 || us < least) {
      least = us;
      best = v;
    }
  }
  return best;
}

// the index of the tile in its table (tall: rows of A lie so that 320 of them are within 32-bit offsets)
static int choose(int ta, int tw, bool ragged, bool tall, int M, int N, int nk, int groups, bool by_rows, bool gated) {
  if (ta == 1)
    return ragged ? 1 + pick_tile(TILES + 1, 6, PART, M, N, nk, groups, by_rows, gated) : pick_tile(TILES, tall ? 14 : 12, PART, M, N, nk, groups, by_rows, gated);
  return tw == 1 ? pick_tile(TILES_MIXED, 5, PART, M, N, nk, groups, by_rows, gated) : pick_tile(TILES_F32, 7, 1.f, M, N, nk, groups, by_rows, gated);
}

extern "C" int fls_seq_gemm_tile_of(int ta, int tw, int M, int N, int K, int groups, int by_rows, int gated) {
  return choose(ta, tw, false, true, M, N, K * (tw == 1 ? 2 : 4) / 128, groups, by_rows != 0, gated != 0);
}

int seq_gemm_tile(const void* A, int ta, const void* W, int tw, void* C, const Epi& epi, int M, int N, int K, int lda, int ldw, int ldc, int groups,
                  const int* offs, const int* a_rows, long long a_gs, int a_mod, long long w_gs, long long c_gs, hipStream_t s) {
  const int ea = ta == 1 ? 2 : 4, ew = tw == 1 ? 2 : 4;
  // Whole K tiles; stores of four columns, or of one for a plain product of up to 128 columns (a router of 10 outputs
  // over the rows of 9 prompts of 1,500 tokens: 76 us from the kernel for any shape, 15 here); 32-bit offsets within a tile.
  const bool ragged = N % 4 || ldc % 4 || (uintptr_t)C % 16 || (offs == nullptr && c_gs % 4) || (epi.bias != nullptr && (uintptr_t)epi.bias % 16);
  if (K * ew % 128 || (ragged && (epi.kind != 0 || epi.bias != nullptr || offs != nullptr || groups != 1 || N > 128))) return 0;
  if (((long long)lda * 256 + K) * ea >= (1LL << 31) || ((long long)ldw * 256 + K) * ew >= (1LL << 31)) return 0;
  if (offs == nullptr && groups > 65535) return 0;
  const bool gated = epi.kind >= EPI_GATE;
  if (gated && (N % 8 || (long long)N * ldw * ew >= (1LL << 31) || (offs == nullptr && groups > 1))) return 0;
  if (a_rows != nullptr && (long long)M * lda * ea >= (1LL << 31)) return 0;      // (there are at most as many rows of A as of the product)
  const int nk = K * ew / 128;
  const Tile t = {(const char*)A, (const char*)W, C, epi, M, N, nk, lda * ea, ldw * ew, ldc, a_rows, offs, groups, w_gs * ew, a_gs * ea, c_gs,
                  a_mod < 1 ? 1 : a_mod, 0, 0, 0, ragged};
  const int tile = choose(ta, tw, ragged, ((long long)lda * 320 + K) * ea < (1LL << 31), M, N, nk, groups, offs != nullptr, gated);
  if (ta == 1) {
    switch (tile) {
      case 0: return start<gemm_tile_big<8>>(256, 256, 256, t256::lds_bytes(8), t, s);
      case 1: return start<gemm_tile_mid<bf16_t, bf16_t, 4, 4, 2, 2, 1>>(128, 128, 256, 2 * 32768, t, s);
      case 2: return start<gemm_tile_mid<bf16_t, bf16_t, 4, 4, 2, 1, 2>>(128, 128, 512, 4 * 32768, t, s);
      case 3: return start<gemm_tile_mid<bf16_t, bf16_t, 2, 4, 3, 1, 2>>(64, 128, 512, 6 * 24576, t, s);
      case 4: return start<gemm_tile_mid<bf16_t, bf16_t, 2, 2, 4, 1, 2>>(64, 64, 512, 8 * 16384, t, s);
      case 5: return start<gemm_tile_mid<bf16_t, bf16_t, 1, 2, 3, 1, 4>>(32, 64, 1024, 12 * 12288, t, s);
      case 6: return start<gemm_tile_mid<bf16_t, bf16_t, 1, 1, 4, 1, 4>>(32, 32, 1024, 16 * 8192, t, s);
      case 7: return start<gemm_tile_big<6>>(192, 256, 256, t256::lds_bytes(6), t, s);
      case 8: return start<gemm_tile_big<4>>(128, 256, 256, t256::lds_bytes(4), t, s);
      case 10: return start<gemm_tile_big<5>>(160, 256, 256, t256::lds_bytes(5), t, s);
      case 11: return start<gemm_tile_big<7>>(224, 256, 256, t256::lds_bytes(7), t, s);
      case 12: return start<gemm_tile_big<9>>(288, 256, 256, t256::lds_bytes(9), t, s);
      case 13: return start<gemm_tile_big<10>>(320, 256, 256, t256::lds_bytes(10), t, s);
      default: return start<gemm_tile_mid<bf16_t, bf16_t, 2, 4, 3, 2, 1>>(64, 128, 256, 3 * 24576, t, s);
    }
  }
  if (tw == 1) {
    switch (tile) {
      case 0: return start<gemm_tile_mid<float, bf16_t, 2, 4, 2, 2, 1>>(64, 128, 256, 2 * 32768, t, s);
      case 1: return start<gemm_tile_mid<float, bf16_t, 2, 4, 2, 1, 2>>(64, 128, 512, 4 * 32768, t, s);
      case 2: return start<gemm_tile_mid<float, bf16_t, 2, 2, 3, 1, 2>>(64, 64, 512, 6 * 24576, t, s);
      case 3: return start<gemm_tile_mid<float, bf16_t, 2, 2, 3, 2, 1>>(64, 64, 256, 3 * 24576, t, s);
      default: return start<gemm_tile_mid<float, bf16_t, 1, 1, 3, 1, 4>>(32, 32, 1024, 12 * 12288, t, s);
    }
  }
  switch (tile) {
    case 0: return start<gemm_tile_mid<float, float, 4, 4, 2, 2, 1>>(128, 128, 256, 2 * 32768, t, s);
    case 1: return start<gemm_tile_mid<float, float, 4, 4, 2, 1, 2>>(128, 128, 512, 4 * 32768, t, s);
    case 2: return start<gemm_tile_mid<float, float, 2, 4, 3, 1, 2>>(64, 128, 512, 6 * 24576, t, s);
    case 3: return start<gemm_tile_mid<float, float, 2, 2, 4, 1, 2>>(64, 64, 512, 8 * 16384, t, s);
    case 4: return start<gemm_tile_mid<float, float, 1, 2, 3, 1, 4>>(32, 64, 1024, 12 * 12288, t, s);
    case 6: return start<gemm_tile_mid<float, float, 2, 2, 3, 3, 1>>(64, 64, 256, 3 * 16384, t, s);
    default: return start<gemm_tile_mid<float, float, 1, 1, 4, 1, 4>>(32, 32, 1024, 16 * 8192, t, s);
  }
}
