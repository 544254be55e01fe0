// The delta rules of delta.hip and gated_delta.hip for steps with many rows per request, 16 rows (a chunk) at a time on the fp32
// matrix cores.  With S the state before a chunk and V its 16 value rows both rules have the form
//
//   X = M1 S + N1 V,     O = Q+ S + B X (+ Bk V),     S' = diag(P) S + L1^T X (+ L2^T V)
//
//   gated:        X = the updates u;                M1 = -(I + b A)^-1 b K+,   N1 = (I + b A)^-1 b
//   generalized:  X = k^T S before each row;        M1 = (I + A)^-1 K+,        N1 = (I + A)^-1 Ak
//
// (in brackets the generalized rule's) where K+, Q+ are rows times the decay since the chunk's start, and A, B, .. hold
// sum_i left_t,i right_s,i prod(decays between s and t) for s < t (B: and s = t).  Two kernels:
//
//   factors (independent of the state, a block per chunk and head)     M1 .. into memory.  Nothing divides by a decay: a pair (t, s)
//     belongs to the one of four levels (8, 4, 2, 1) at which t is in the upper and s in the lower half of the same block of rows; left
//     rows carry the decay from the middle to t, right rows from s to the middle, both at most 1, and one wave's MFMAs make a
//     level's products.  The triangular system is solved by a thread per column.  Products of decays are made in fp64 and rounded once.
//   walk (a wave per 16 value columns, head and request)     three products a chunk.  An accumulator's layout of the 16x16x4 MFMA is the
//     layout of its right operand when lane group g holds elements 4 g .. 4 g + 3 of 16 and MFMA r multiplies the r-th ones: S and X go
//     from product to product in registers, without LDS, barriers or shuffles.  The next chunk's factors are loaded as
//     soon as this chunk's have been used.
//
// What bounds the row-by-row forms is a chain of LDS reads, sums over lanes and updates per row, 0.5 us (128 x 128) or 0.7 us (64 x 64); a
// chunk's chain here is its MFMAs and the two kernels' traffic over the factors, which stay in the last-level cache for as many chunks
// as are made at a time.  Row by row against this (16 heads; outputs' norm included), gated 128 x 128 and generalized 64 x 64:
//   1 request of 2048 rows:  640 -> 388 us, 1590 -> 290 us       9 of 1500:  1060 -> 702 us, 1410 -> 410 us
// Error against 64 bits (2-norm; 1500 rows of 64 x 64, 700 of 128 x 128), row by row and here: gated outputs 1.13e-7 and 1.12e-7 with strong
// decays, 1.67e-7 .. 1.69e-7 and 1.51e-7 .. 1.54e-7 with weak ones, generalized 1.83e-7 .. 1.88e-7 and 1.65e-7 .. 1.69e-7; states 0.58e-7 .. 1.66e-7
// and 0.54e-7 .. 1.37e-7.  It takes sums of 16 terms joined by trees, decays rounded once, a state that is rounded once a chunk and
// (gated) diagonals outside the MFMAs; without these it was up to 13% above the rows' (and 3% faster).
#include "seq_common.h"
#include "fls_seq.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
#define CH 16

__device__ __forceinline__ floatx4 mfma16(const floatx4& a, const floatx4& b, floatx4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}

// a chunk's factors of one head: M1, Q+ [16][D], L1, (generalized) L2 [D][16], N1, B, (generalized) Bk [16][16], P [D].  The matrices lie as the walk's
// waves read them, 16 x 16 at a time as left operands: lane (row % 16, group g) its elements 4 g .. 4 g + 3, 1 KB in a row
template <int D, bool GEN>
struct Lay {
  static constexpr int QP = CH * D, L1 = 2 * CH * D, L2 = 3 * CH * D, N1 = (GEN ? 4 : 3) * CH * D, B = N1 + CH * CH, BK = B + CH * CH,
                       P = GEN ? BK + CH * CH : BK, SIZE = P + D;
};

__device__ __forceinline__ int frag(int row, int k) { return (k >> 2) * 64 + row * 4 + (k & 3); }

struct Delta {
  const float* q;          // queries (gated) or r
  int ldq;
  const float* k;
  int ldk;
  const float* v;
  int ldv;
  const float* dec;        // gated: decays; generalized: wz
  int ldd;
  const float* rate;       // gated: beta [T, H]; generalized: az
  int ldr;
  const float* w0;         // generalized only
  float* state;
  float* raw;              // [T, H dv]
  float* fac;
  const int *cu, *pos0, *slot;
  int H, rep, dv;          // rep: heads that share q and k
  float q_scale, eps, decay_scale;
  int c0, nc;              // this launch's chunks of every request: c0 .. c0 + nc - 1
};

template <int D, bool GEN>
__global__ __launch_bounds__(256, GEN ? 2 : 3) void delta_factors_kernel(Delta a) {
  using L = Lay<D, GEN>;
  constexpr int LD = D + 4, M = D / 64, PARTS = 256 / D;
  __shared__ __attribute__((aligned(16))) float K[CH * LD], Q[CH * LD], G[CH * LD], R[GEN ? CH * LD : 4], Z[3][CH * LD];
  __shared__ __attribute__((aligned(16))) float A[CH][CH], B[CH][CH], Ak[GEN ? CH : 1][CH], Bk[GEN ? CH : 1][CH];
  __shared__ float sb[CH];
  const int s = blockIdx.z, h = blockIdx.y, cl = blockIdx.x;
  const int r0 = a.cu[s] + (a.c0 + cl) * CH, end = a.cu[s + 1];
  if (r0 >= end) return;
  float* fac = a.fac + (((size_t)cl * gridDim.z + s) * a.H + h) * L::SIZE;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  {                                                           // sixteen threads a row; rows past the request's end change nothing
    const int row = tid >> 4, n = tid & 15, t = r0 + row;
    const bool ok = t < end;
    floatx4 q[M], k[M], g[M], r[M];
    float qq = 0.f, kk = 0.f, qk = 0.f, qr = 0.f;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int i = 64 * m + 4 * n;
      q[m] = k[m] = r[m] = floatx4{0.f, 0.f, 0.f, 0.f};
      g[m] = floatx4{1.f, 1.f, 1.f, 1.f};
      if (ok) {
        q[m] = *reinterpret_cast<const floatx4*>(a.q + (size_t)t * a.ldq + (size_t)(h / a.rep) * D + i);
        k[m] = *reinterpret_cast<const floatx4*>(a.k + (size_t)t * a.ldk + (size_t)(h / a.rep) * D + i);
        g[m] = *reinterpret_cast<const floatx4*>(a.dec + (size_t)t * a.ldd + (size_t)h * D + i);
        if constexpr (GEN) {
          const floatx4 az = *reinterpret_cast<const floatx4*>(a.rate + (size_t)t * a.ldr + (size_t)h * D + i);
          const floatx4 w0 = *reinterpret_cast<const floatx4*>(a.w0 + (size_t)h * D + i);
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            g[m][x] = expf(-a.decay_scale * sigmoid_f(g[m][x] + w0[x]));
            r[m][x] = sigmoid_f(az[x]) * k[m][x];
          }
        }
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        qq += q[m][x] * q[m][x]; kk += k[m][x] * k[m][x]; qk += q[m][x] * k[m][x]; qr += q[m][x] * r[m][x];
      }
    }
    qq = row16_sum(qq); kk = row16_sum(kk); qk = row16_sum(qk); qr = row16_sum(qr);
    float fq = 1.f, fk = 1.f, fr = 1.f;
    if constexpr (GEN) fr = 1.f / (kk + a.eps);
    else { fq = a.q_scale / sqrtf(qq + a.eps); fk = 1.f / sqrtf(kk + a.eps); }
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int i = row * LD + 64 * m + 4 * n;
      *reinterpret_cast<floatx4*>(Q + i) = q[m] * fq;
      *reinterpret_cast<floatx4*>(K + i) = k[m] * fk;
      *reinterpret_cast<floatx4*>(G + i) = g[m];
      if constexpr (GEN) *reinterpret_cast<floatx4*>(R + i) = r[m] * fr;
    }
    if (n == 0 && !GEN) sb[row] = ok ? sigmoid_f(a.rate[(size_t)t * a.ldr + h]) : 0.f;
    // (the diagonals: no decay between a row and itself; above them nothing)
    if (n >= row) {
      A[row][n] = 0.f;
      B[row][n] = n > row ? 0.f : GEN ? qr * fr : qk * fq * fk;
      if constexpr (GEN) { Ak[row][n] = 0.f; Bk[row][n] = n > row ? 0.f : qk; }
    }
  }
  __syncthreads();
  const int ch = tid % D, part = tid / D;                     // a channel a thread
  float kp[CH];                                               // (the last part's threads: this channel's decayed keys)
  {
    float g[CH];
#pragma unroll
    for (int t = 0; t < CH; ++t) g[t] = G[t * LD + ch];
#pragma unroll
    for (int l = 0; l < 3; ++l) {                             // (the last level is the rows' own decays)
      if (part != (D == 128 ? 0 : l)) continue;
      const int b = 8 >> l;
#pragma unroll
      for (int m0 = 0; m0 < CH; m0 += 2 * b) {
        double z = 1.0;
#pragma unroll
        for (int t = m0 + b; t < m0 + 2 * b; ++t) { z *= g[t]; Z[l][t * LD + ch] = (float)z; }
        z = 1.0;
#pragma unroll
        for (int t = m0 + b - 1; t >= m0; --t) { Z[l][t * LD + ch] = (float)z; z *= g[t]; }
      }
    }
    if (part == PARTS - 1) {
      double z = 1.0;
#pragma unroll
      for (int t = 0; t < CH; ++t) {
        const double before = z;
        z *= g[t];
        kp[t] = (float)(K[t * LD + ch] * (GEN ? before : z));
        fac[L::QP + (ch >> 4) * 256 + frag(t, ch & 15)] = (float)(Q[t * LD + ch] * z);
      }
      fac[L::P + ch] = (float)z;
      z = 1.0;
      floatx4 l1[4], l2[4];
#pragma unroll
      for (int t = CH - 1; t >= 0; --t) {
        const float k = (float)(K[t * LD + ch] * z);
        l2[t >> 2][t & 3] = k;
        if constexpr (GEN) l1[t >> 2][t & 3] = (float)(-R[t * LD + ch] * z);
        z *= g[t];
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        *reinterpret_cast<floatx4*>(fac + L::L1 + (ch >> 4) * 256 + frag(ch & 15, 4 * x)) = GEN ? l1[x] : l2[x];
        if constexpr (GEN) *reinterpret_cast<floatx4*>(fac + L::L2 + (ch >> 4) * 256 + frag(ch & 15, 4 * x)) = l2[x];
      }
    }
  }
  __syncthreads();
  {                                                           // wave = level: pairs whose highest differing bit is b
    const int fr = lane & 15, grp = lane >> 4, b = 8 >> wave;
    const bool up = (fr & b) != 0, first = (fr & (b - 1)) == 0;
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f}, one = {1.f, 1.f, 1.f, 1.f};
    constexpr int J = D / 16;
    floatx4 sA[J], sB[J], sAk[J], sBk[J];
#pragma unroll
    for (int j = 0; j < J; ++j) sA[j] = sB[j] = sAk[j] = sBk[j] = zero;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int e = fr * LD + 16 * j + 4 * grp;
      floatx4 &accA = sA[j], &accB = sB[j], &accAk = sAk[j], &accBk = sBk[j];
      const floatx4 z = wave < 3 ? *reinterpret_cast<const floatx4*>(&Z[wave][e]) : up ? *reinterpret_cast<const floatx4*>(G + e) : one, k = *reinterpret_cast<const floatx4*>(K + e),
                    q = *reinterpret_cast<const floatx4*>(Q + e);
      if constexpr (GEN) {
        const floatx4 zx = first ? one : *reinterpret_cast<const floatx4*>(&Z[wave][up ? e - LD : e]);     // (X reads the state before its row's decay)
        const floatx4 r = *reinterpret_cast<const floatx4*>(R + e);
        const floatx4 la = up ? k * zx : zero, lb = up ? q * z : zero, ra = up ? zero : r * z, rb = up ? zero : k * z;
        accA = mfma16(la, ra, accA);
        accAk = mfma16(la, rb, accAk);
        accB = mfma16(lb, ra, accB);
        accBk = mfma16(lb, rb, accBk);
      } else {
        const floatx4 kz = k * z, la = up ? kz : zero, lb = up ? q * z : zero, ra = up ? zero : kz;
        accA = mfma16(la, ra, accA);
        accB = mfma16(lb, ra, accB);
      }
    }
#pragma unroll
    for (int d = J / 2; d > 0; d /= 2)
#pragma unroll
      for (int j = 0; j < d; ++j) { sA[j] += sA[j + d]; sB[j] += sB[j + d]; sAk[j] += sAk[j + d]; sBk[j] += sBk[j + d]; }
    const floatx4 accA = sA[0], accB = sB[0], accAk = sAk[0], accBk = sBk[0];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 4 * grp + r;
      if (((t ^ fr) & ~(2 * b - 1)) == 0 && (t & b) != 0 && (fr & b) == 0) {
        A[t][fr] = GEN ? accA[r] : accA[r] * sb[t];
        B[t][fr] = accB[r];
        if constexpr (GEN) { Ak[t][fr] = accAk[r]; Bk[t][fr] = accBk[r]; }
      }
    }
  }
  __syncthreads();
  {
    const int t = tid >> 4, u = tid & 15;
    fac[L::B + frag(t, u)] = GEN ? -B[t][u] : B[t][u];
    if constexpr (GEN) fac[L::BK + frag(t, u)] = Bk[t][u];
  }
  // a column a thread: the last part's threads a channel of M1, the first sixteen a column of N1
  const bool isn = tid < CH;
  if (part == PARTS - 1 || isn) {
    float x[CH];
    float* o = fac + (isn ? L::N1 : (ch >> 4) * 256) + frag(0, ch & 15);
#pragma unroll
    for (int t = 0; t < CH; ++t) {
      float rhs;
      if constexpr (GEN) rhs = isn ? Ak[t][tid & 15] : kp[t];
      else rhs = sb[t] * (isn ? (t == tid ? 1.f : 0.f) : -kp[t]);
#pragma unroll
      for (int u = 0; u < t; ++u) rhs -= A[t][u] * x[u];
      x[t] = rhs;
      o[4 * t] = rhs;
    }
  }
}

// A chunk's lower triangular matrix (m: where it lies in LDS, f: as a left operand) times 16 rows of which some are not finite: those
// rows reach the rows after them (DIAG: and their own) only.
template <bool DIAG>
__device__ __forceinline__ floatx4 below(const float* m, const floatx4& f, const floatx4& v) {
  const int lane = threadIdx.x & 63, fr = lane & 15, grp = lane >> 4;
  floatx4 c;
#pragma unroll
  for (int r = 0; r < 4; ++r) c[r] = __builtin_isfinite(v[r]) ? v[r] : 0.f;
  floatx4 acc = mfma16(f, c, floatx4{0.f, 0.f, 0.f, 0.f});
#pragma unroll 1
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const float e = __shfl(v[x], g * 16 + fr, 64);          // row 4 g + x of this lane's column
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 4 * grp + r, s = 4 * g + x;
        if (!__builtin_isfinite(e) && (DIAG ? t >= s : t > s)) acc[r] += m[frag(t, s)] * e;
      }
    }
  return acc;
}

// wave = 16 value columns of one head and request; the block's waves share the factors, which travel to LDS a chunk ahead
template <int D, bool GEN>
__global__ __launch_bounds__(256, 2) void delta_walk_kernel(Delta a) {
  using L = Lay<D, GEN>;
  constexpr int J = D / 16, NL = (L::SIZE + 1023) / 1024, BUF = NL * 1024;       // 4 KB (16 bytes a thread) at a time
  __shared__ __attribute__((aligned(16))) float fs[2][BUF];
  const int h = blockIdx.x, s = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), fr = lane & 15, grp = lane >> 4;
  const int col = (blockIdx.z * 4 + wave) * 16 + fr;
  const bool live = (int)(blockIdx.z * 4 + wave) * 16 < a.dv;  // (dv is a multiple of 16: whole waves; the others only help to load)
  const int start = a.cu[s], end = a.cu[s + 1];
  const int first = start + a.c0 * CH;
  if (first >= end) return;
  const int stop = min(end, first + a.nc * CH);
  const int si = GEN ? a.dv : 1, sc = GEN ? 1 : D;            // strides of the state's key channels and value columns
  float* sp = a.state + ((size_t)a.slot[s] * a.H + h) * D * a.dv + (size_t)(live ? col : 0) * sc;
  const float* vp = a.v + (size_t)h * a.dv + (live ? col : 0);
  float* op = a.raw + (size_t)h * a.dv + (live ? col : 0);
  const size_t ldo = (size_t)a.H * a.dv;
  // (the descriptor ends with the factors: the last load's threads past them write zeros)
  const size_t fstep = (size_t)gridDim.y * a.H * L::SIZE;
  const float* f = a.fac + ((size_t)s * a.H + h) * L::SIZE;
  auto fetch = [&](int buf) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(f), (short)0, L::SIZE * 4, 0x00020000);
#pragma unroll
    for (int i = 0; i < NL; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(fs[buf] + i * 1024 + wave * 256), 16,
                                               lane * 16, i * 4096 + wave * 1024, 0, 0);
    f += fstep;
  };
  fetch(0);
  floatx4 vn, O = {0.f, 0.f, 0.f, 0.f};
  auto load_v = [&](int row) {
#pragma unroll
    for (int r = 0; r < 4; ++r) vn[r] = live && row + 4 * grp + r < end ? vp[(size_t)(row + 4 * grp + r) * a.ldv] : 0.f;
  };
  auto store_o = [&](int row) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (live && row + 4 * grp + r < end) op[(size_t)(row + 4 * grp + r) * ldo] = O[r];
  };
  load_v(first);
  floatx4 S[J];
  const bool carried = a.pos0[s] > 0 || a.c0 > 0;
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[j][r] = carried ? sp[(size_t)(16 * j + 4 * grp + r) * si] : 0.f;
  int buf = 0;
  for (int r0 = first; r0 < stop; r0 += CH, buf ^= 1) {
    const floatx4 v = vn, zero = {0.f, 0.f, 0.f, 0.f};
    // (a builtin, which the compiler counts: behind the same wait in asm it believed the state's registers, loaded in front of the loop, still on their
    // way and had each chunk wait for half of the next one's factors before its first product)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x70);                                  // vmcnt(0) lgkmcnt(0): this wave's part of the chunk's factors is here ...
    __builtin_amdgcn_s_barrier();                                      // ... and everybody's; the other buffer has been read
    asm volatile("" ::: "memory");
    if (r0 > first) store_o(r0 - CH);
    if (r0 + CH < stop) { fetch(buf ^ 1); load_v(r0 + CH); }
    if (!live) continue;
    const float* F = fs[buf] + lane * 4;
    const auto at = [&](int off) { return *reinterpret_cast<const floatx4*>(F + off); };
    // (each product's operands are read from LDS while the one before runs: the barriers keep the reads where they stand)
    floatx4 m1[J], qp[J], l1[J], l2[GEN ? J : 1];
    // (gated: N1 and B without their diagonals, which enter by a multiply-add of their own.  They are the largest terms where decays are
    // strong, and a MFMA rounds each product)
    const auto lower = [&](int off) {
      floatx4 m = at(off);
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] = 4 * grp + r == fr ? 0.f : m[r];
      return m;
    };
    const auto add_diagonal = [&](int off, const floatx4& y, floatx4 c) {      // of this lane's rows 4 grp + r
#pragma unroll
      for (int r = 0; r < 4; ++r) c[r] = __builtin_fmaf(fs[buf][off + frag(4 * grp + r, 4 * grp + r)], y[r], c[r]);
      return c;
    };
    const floatx4 n1 = GEN ? at(L::N1) : lower(L::N1), b = GEN ? at(L::B) : lower(L::B), bk = GEN ? at(L::BK) : zero;
#pragma unroll
    for (int j = 0; j < J; ++j) m1[j] = at(256 * j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < J; ++j) qp[j] = at(L::QP + 256 * j);
    floatx4 X, x[J], o[J];                                     // (short sums, then a tree, like the row-by-row kernels' sums over lanes)
#pragma unroll
    for (int j = 0; j < J; ++j) x[j] = mfma16(m1[j], S[j], zero);
    X = mfma16(n1, v, zero);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      l1[j] = at(L::L1 + 256 * j);
      if constexpr (GEN) l2[j] = at(L::L2 + 256 * j);
    }
#pragma unroll
    for (int j = 0; j < J; ++j) o[j] = mfma16(qp[j], S[j], zero);
#pragma unroll
    for (int d = J / 2; d > 0; d /= 2)
#pragma unroll
      for (int j = 0; j < d; ++j) { x[j] += x[j + d]; o[j] += o[j + d]; }
    X += x[0];
    if constexpr (GEN) {
      O = mfma16(b, X, zero) + (mfma16(bk, v, zero) + o[0]);
    } else {
      X = add_diagonal(L::N1, v, X);
      O = add_diagonal(L::B, X, mfma16(b, X, zero) + o[0]);
    }
    bool odd = false;                                          // (zeros above the diagonals would spread a later row's inf or NaN)
#pragma unroll
    for (int r = 0; r < 4; ++r) odd |= !__builtin_isfinite(v[r]) | !__builtin_isfinite(X[r]);
    if (__any(odd)) {
      X = below<false>(fs[buf] + L::N1, n1, v) + x[0];         // (GEN: N1 has no diagonal)
      if constexpr (GEN) {
        O = below<true>(fs[buf] + L::B, b, X) + (below<true>(fs[buf] + L::BK, bk, v) + o[0]);
      } else {
        X = add_diagonal(L::N1, v, X);
        O = add_diagonal(L::B, X, below<false>(fs[buf] + L::B, b, X) + o[0]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < J; ++j) {                              // (the chunk's sum first: one rounding at the state's size)
      const floatx4 P = *reinterpret_cast<const floatx4*>(fs[buf] + L::P + 16 * j + 4 * grp);
      floatx4 u = mfma16(l1[j], X, zero);
      if constexpr (GEN) u = mfma16(l2[j], v, u);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[j][r] = __builtin_fmaf(S[j][r], P[r], u[r]);
    }
  }
  if (!live) return;
  store_o(start + (stop - 1 - start) / CH * CH);
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) sp[(size_t)(16 * j + 4 * grp + r) * si] = S[j][r];
}

template <int D, bool GEN>
int run(Delta a, int B, int max_rows, int seg, hipStream_t st) {
  const int chunks = (max_rows + CH - 1) / CH;
  for (a.c0 = 0; a.c0 < chunks; a.c0 += seg) {
    a.nc = chunks - a.c0 < seg ? chunks - a.c0 : seg;
    hipLaunchKernelGGL((delta_factors_kernel<D, GEN>), dim3(a.nc, a.H, B), dim3(256), 0, st, a);
    SEQ_LAUNCH_CHECK();
    hipLaunchKernelGGL((delta_walk_kernel<D, GEN>), dim3(a.H, B, (a.dv + 63) / 64), dim3(256), 0, st, a);
    SEQ_LAUNCH_CHECK();
  }
  return 0;
}

}  // namespace

// fac: B H seg * (49 d + 512) floats.  Rows of raw are finished by the caller.  Returns -2 for head sizes or alignments not served.
int seq_gated_delta_chunked(const float* qkv, int ldq, const float* beta, int ldb, const float* decay, int ldd, float* state, float* raw,
                            const int* cu, const int* pos0, const int* slot, int B, int H, int G, int d, int dv, float q_scale,
                            float unit_eps, int max_rows, float* fac, int seg, fls_stream_t s) {
  if ((d != 64 && d != 128) || dv % 16 || ldq % 4 || ldd % 4 || (uintptr_t)qkv % 16 || (uintptr_t)decay % 16 || (uintptr_t)fac % 16 ||
      seg < 1 || B > 65535 || H > 65535)
    return -2;
  Delta a = {};
  a.q = qkv; a.ldq = ldq; a.k = qkv + (size_t)G * d; a.ldk = ldq; a.v = qkv + (size_t)2 * G * d; a.ldv = ldq;
  a.dec = decay; a.ldd = ldd; a.rate = beta; a.ldr = ldb; a.state = state; a.raw = raw; a.fac = fac;
  a.cu = cu; a.pos0 = pos0; a.slot = slot; a.H = H; a.rep = H / G; a.dv = dv; a.q_scale = q_scale; a.eps = unit_eps;
  return d == 64 ? run<64, false>(a, B, max_rows, seg, (hipStream_t)s) : run<128, false>(a, B, max_rows, seg, (hipStream_t)s);
}

// fac: B H seg * (65 d + 768) floats
int seq_delta_rule_chunked(const float* r, int ldr, const float* k, int ldk, const float* v, int ldv, const float* az, int lda,
                           const float* wz, int ldw, const float* w0, float* state, float* raw, const int* cu, const int* pos0,
                           const int* slot, int B, int H, int d, float decay_scale, float key_eps, int max_rows, float* fac, int seg,
                           fls_stream_t s) {
  if ((d != 64 && d != 128) || ldr % 4 || ldk % 4 || lda % 4 || ldw % 4 || (uintptr_t)r % 16 || (uintptr_t)k % 16 || (uintptr_t)az % 16 ||
      (uintptr_t)wz % 16 || (uintptr_t)w0 % 16 || (uintptr_t)fac % 16 || seg < 1 || B > 65535 || H > 65535)
    return -2;
  Delta a = {};
  a.q = r; a.ldq = ldr; a.k = k; a.ldk = ldk; a.v = v; a.ldv = ldv; a.dec = wz; a.ldd = ldw; a.rate = az; a.ldr = lda; a.w0 = w0;
  a.state = state; a.raw = raw; a.fac = fac; a.cu = cu; a.pos0 = pos0; a.slot = slot; a.H = H; a.rep = 1; a.dv = d;
  a.eps = key_eps; a.decay_scale = decay_scale;
  return d == 64 ? run<64, true>(a, B, max_rows, seg, (hipStream_t)s) : run<128, true>(a, B, max_rows, seg, (hipStream_t)s);
}
