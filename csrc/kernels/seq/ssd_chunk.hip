// The selective state-space scan of scan.hip for steps with many rows per request, 64 rows (a chunk) at a time on the fp32
// matrix cores.  With la_t = -exp(A) dt_t, c_i = la_1 + .. + la_i inside a chunk and S the state before it:
//
//   y_i = exp(c_i) C_i . S + sum_{j <= i} exp(c_i - c_j) dt_j (C_i . B_j) x_j,    S' = exp(c_64) S + sum_j exp(c_64 - c_j) dt_j B_j x_j^T
//
// so a request of n rows is a chain of n / 64 chunks instead of n rows.  What bounds the row-by-row form is that chain (0.7 us a
// row); here it is a chunk's chain of products and LDS reads, with C, the scores and z loaded while the chunk is laid down.  C_i . B_j
// is the same for all heads of a group: a first kernel leaves it in memory once ([T, groups, 64] fp32).  Row by row against this, heads
// of 64 x 128: 2 requests of 512 rows, 32 heads 350 -> 63 us; 8 of 2048 rows, 64 heads 1880 -> 676; 1 of 2048 1443 -> 197.  Exponents
// are differences of running sums: the sums are fp64, so a difference is exact to fp32 however far a chunk has decayed.
// Error against 64 bits (2-norm, row by row and here): outputs 1.39e-7 and 1.34e-7, states 1.03e-7 and 0.97e-7 where a row decays by some 0.85;
// 1.26e-7 and 1.23e-7, 0.78e-7 and 0.89e-7 by 0.6; 12e-7 and 1.8e-7, 14e-7 and 1.3e-7 by 0.99.  It takes sums of 16 or 32 terms joined
// by trees and a row's own term outside the MFMAs, which round each product: in single chains outputs were up to 1.8 times as far off.
// All products are fp32 (16x16x4 MFMAs: lane group g holds elements 4 g .. 4 g + 3 of 16, MFMA r multiplies the r-th ones).
#include "seq_common.h"
#include "fls_seq.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
#define CQ 64

__device__ __forceinline__ floatx4 mfma16(const floatx4& a, const floatx4& b, floatx4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}

struct Ssd {
  const float* xbc;
  int ldx;
  const float* z;
  int ldz;
  const float* dt;
  int lddt;
  const float *dt_bias, *A_log, *Dskip;
  float* state;
  float* out;
  int ldo;
  const int *cu, *pos0, *slot;
  int nh, P, N, G;
  float* scores;       // [T, G, 64]: C_i . B_j of row i and row j of its chunk, j <= i
};

// block = (chunk, group, request), wave = 16 of its rows
template <int N>
__global__ __launch_bounds__(256) void ssd_scores_kernel(Ssd a) {
  const int s = blockIdx.z, g = blockIdx.y;
  const int r0 = a.cu[s] + blockIdx.x * CQ, end = a.cu[s + 1];
  if (r0 >= end) return;
  const int nt = min(CQ, end - r0);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, fr = lane & 15, grp = lane >> 4;
  const int i0 = 16 * w;
  if (i0 >= nt) return;
  const int inner = a.nh * a.P;
  const float* B = a.xbc + (size_t)r0 * a.ldx + inner + g * a.N;
  const float* C = B + a.G * a.N;
  const float* crow = C + (size_t)min(i0 + fr, nt - 1) * a.ldx + 4 * grp;
  // (sums of 16 terms, then a tree)
  floatx4 part[N / 16][4];
#pragma unroll
  for (int q = 0; q < N / 16; ++q) {
    const floatx4 c = *reinterpret_cast<const floatx4*>(crow + 16 * q);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      part[q][j] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (j > w) continue;
      const floatx4 b = *reinterpret_cast<const floatx4*>(B + (size_t)min(16 * j + fr, nt - 1) * a.ldx + 4 * grp + 16 * q);
      part[q][j] = mfma16(c, b, part[q][j]);
    }
  }
#pragma unroll
  for (int d = N / 32; d > 0; d /= 2)
#pragma unroll
    for (int q = 0; q < d; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) part[q][j] += part[q + d][j];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (j > w) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + 4 * grp + r;
      if (i < nt) a.scores[((size_t)(r0 + i) * a.G + g) * CQ + 16 * j + fr] = part[0][j][r];
    }
  }
}

// block = (16 PT value columns, head, request), walking the request's chunks; wave w: rows 16 w .. of y, state rows 16 NW w ..
// (N = 64 NW).  The state stays in registers where it is summed and in LDS where the next chunk's y reads it.
template <int PT, int NW>
__global__ __launch_bounds__(256, 2) void ssd_chunk_kernel(Ssd a) {
  constexpr int N = 64 * NW, LB = N + 4, LX = 16 * PT + 4;     // (row strides that put lane groups 16 banks apart)
  __shared__ __attribute__((aligned(16))) float Bs[CQ * LB];
  __shared__ __attribute__((aligned(16))) float xs[CQ * LX];
  __shared__ float Ss[N * LX];
  __shared__ double cs[CQ];
  __shared__ float dts[CQ], wj[CQ], self[CQ];                 // self: a row's own term of y, D's among it
  const int s = blockIdx.z, h = blockIdx.y, p0 = blockIdx.x * 16 * PT;
  const int g = h / (a.nh / a.G), inner = a.nh * a.P;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, fr = lane & 15, grp = lane >> 4;
  const int a0 = a.cu[s], a1 = a.cu[s + 1];
  const float negA = -expf(a.A_log[h]), db = a.dt_bias[h], dsk = a.Dskip[h];
  float* sp = a.state + (((size_t)a.slot[s] * a.nh + h) * N) * a.P + p0;
  const bool carried = a.pos0[s] > 0;
  floatx4 S[NW][PT];
#pragma unroll
  for (int k = 0; k < NW; ++k)
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = 16 * (NW * w + k) + 4 * grp + r;
        S[k][p][r] = carried ? sp[(size_t)n * a.P + 16 * p + fr] : 0.f;
      }
  // the next chunk's inputs come into registers while this one is computed
  constexpr int NB4 = CQ * N / 4 / 256, NX4 = (CQ * 16 * PT / 4 + 255) / 256;
  floatx4 pb[NB4], px[NX4];
  float pdt = 0.f, pself = 0.f;
  auto prefetch = [&](int r0) {
#pragma unroll
    for (int i = 0; i < NB4; ++i) {
      const int e = threadIdx.x + 256 * i, row = e / (N / 4), c = e % (N / 4) * 4;
      pb[i] = r0 + row < a1 ? *reinterpret_cast<const floatx4*>(a.xbc + (size_t)(r0 + row) * a.ldx + inner + g * N + c) : floatx4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < NX4; ++i) {
      const int e = threadIdx.x + 256 * i, row = e / (4 * PT), c = e % (4 * PT) * 4;
      px[i] = r0 + row < a1 ? *reinterpret_cast<const floatx4*>(a.xbc + (size_t)(r0 + row) * a.ldx + h * a.P + p0 + c) : floatx4{0.f, 0.f, 0.f, 0.f};
    }
    if (w == 0) {
      pdt = r0 + lane < a1 ? a.dt[(size_t)(r0 + lane) * a.lddt + h] : 0.f;
      pself = r0 + lane < a1 ? a.scores[((size_t)(r0 + lane) * a.G + g) * CQ + lane] : 0.f;
    }
  };
  prefetch(a0);
  for (int r0 = a0; r0 < a1; r0 += CQ) {
    const int nt = min(CQ, a1 - r0);
    // what this wave's rows of y need beside LDS travels while the chunk is laid down and its decays are summed
    const int row = r0 + min(16 * w + fr, nt - 1);            // (rows past the end are computed from the last one and not stored)
    constexpr bool AHEAD = PT * NW < 4;                       // (C's row too, where the registers are there: with 2 x 2 it spilled, 882 -> 1140 us)
    floatx4 cr[AHEAD ? N / 16 : 1], sr[4];
    float zr[PT][4];
    const float* crow = a.xbc + (size_t)row * a.ldx + inner + (a.G + g) * N + 4 * grp;
    if (16 * w < nt) {
      const float* sc = a.scores + ((size_t)row * a.G + g) * CQ + 4 * grp;
      if constexpr (AHEAD) {
#pragma unroll
        for (int n = 0; n < N / 16; ++n) cr[n] = *reinterpret_cast<const floatx4*>(crow + 16 * n);
      }
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
        if (jb <= w) sr[jb] = *reinterpret_cast<const floatx4*>(sc + 16 * jb);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = min(16 * w + 4 * grp + r, nt - 1);
#pragma unroll
        for (int p = 0; p < PT; ++p) zr[p][r] = a.z[(size_t)(r0 + t) * a.ldz + h * a.P + p0 + 16 * p + fr];
      }
    }
    __syncthreads();                                          // (the chunk before has been read)
#pragma unroll
    for (int i = 0; i < NB4; ++i) {
      const int e = threadIdx.x + 256 * i;
      *reinterpret_cast<floatx4*>(Bs + e / (N / 4) * LB + e % (N / 4) * 4) = pb[i];
    }
#pragma unroll
    for (int i = 0; i < NX4; ++i) {
      const int e = threadIdx.x + 256 * i;
      *reinterpret_cast<floatx4*>(xs + e / (4 * PT) * LX + e % (4 * PT) * 4) = px[i];
    }
#pragma unroll
    for (int k = 0; k < NW; ++k)
#pragma unroll
      for (int p = 0; p < PT; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r) Ss[(16 * (NW * w + k) + 4 * grp + r) * LX + 16 * p + fr] = S[k][p][r];
    if (w == 0) {                                             // a row a lane: step sizes and the running sums of the decays' logarithms
      const float dtv = lane < nt ? softplus_f(pdt + db) : 0.f;
      // (past -104 a row's decay is an exact 0: held at -200 it still is, and no huge or infinite one costs the sums the rows after it)
      double c = lane < nt ? (double)fmaxf(negA * dtv, -200.f) : 0.0;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const double v = __shfl_up(c, o, 64);
        if (lane >= o) c += v;
      }
      const double last = __shfl(c, 63, 64);
      cs[lane] = c;
      dts[lane] = dtv;
      self[lane] = dtv * pself + dsk;
      wj[lane] = expf((float)(last - c)) * dtv;
    }
    __syncthreads();
    if (r0 + CQ < a1) prefetch(r0 + CQ);
    // y: the chunk's earlier rows, then the state before it
    floatx4 own[PT], past[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p) own[p] = past[p] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (16 * w < nt) {
      const int i = 16 * w + fr;
      const double ci = cs[i];
      bool odd = false;                                       // inf or NaN among the wave's own rows
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        if (jb > w) continue;
        const floatx4 m = sr[jb];
        floatx4 l;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * jb + 4 * grp + r;
          l[r] = j < i && j < nt ? expf((float)(ci - cs[j])) * dts[j] * m[r] : 0.f;
        }
#pragma unroll
        for (int p = 0; p < PT; ++p) {
          floatx4 x;
#pragma unroll
          for (int r = 0; r < 4; ++r) x[r] = xs[(16 * jb + 4 * grp + r) * LX + 16 * p + fr];
          if (jb == w) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const bool f = __builtin_isfinite(x[r]);
              odd |= !f;
              x[r] = f ? x[r] : 0.f;
            }
          }
          own[p] = mfma16(l, x, own[p]);
        }
      }
      // (a weight of 0 would spread such a value to the rows before it: it stayed out of the product and makes NaN of its own and
      // later rows; row by row the signs of B and C make inf or NaN of them)
      if (__any(odd)) {
#pragma unroll
        for (int p = 0; p < PT; ++p) {
          int at = CQ;
          for (int j = 15; j >= 0; --j)
            if (!__builtin_isfinite(xs[(16 * w + j) * LX + 16 * p + fr])) at = j;
#pragma unroll
          for (int r = 0; r < 4; ++r) own[p][r] = 4 * grp + r >= at ? __builtin_nanf("") : own[p][r];
        }
      }
      // (sums of 32 terms)
#pragma unroll
      for (int n0 = 0; n0 < N; n0 += 32) {
        floatx4 part[PT];
#pragma unroll
        for (int p = 0; p < PT; ++p) part[p] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int n = n0; n < n0 + 32; n += 16) {
          const floatx4 c = AHEAD ? cr[AHEAD ? n / 16 : 0] : *reinterpret_cast<const floatx4*>(crow + n);
#pragma unroll
          for (int p = 0; p < PT; ++p) {
            floatx4 v;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = Ss[(n + 4 * grp + r) * LX + 16 * p + fr];
            part[p] = mfma16(c, v, part[p]);
          }
        }
#pragma unroll
        for (int p = 0; p < PT; ++p) past[p] += part[p];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * w + 4 * grp + r;
        if (t < nt) {
          const float e = expf((float)cs[t]);
#pragma unroll
          for (int p = 0; p < PT; ++p) {
            const int col = h * a.P + p0 + 16 * p + fr;
            const float y = self[t] * xs[t * LX + 16 * p + fr] + (e * past[p][r] + own[p][r]);
            a.out[(size_t)(r0 + t) * a.ldo + col] = y * silu_f(zr[p][r]);
          }
        }
      }
    }
    // the state after it
    const float dec = expf((float)cs[CQ - 1]);
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      floatx4 u[PT];                                          // (the chunk's sum first, 16 rows at a time: one rounding at the state's size)
#pragma unroll
      for (int p = 0; p < PT; ++p) u[p] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        floatx4 b;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * jb + 4 * grp + r;
          b[r] = Bs[j * LB + 16 * (NW * w + k) + fr] * wj[j];
        }
#pragma unroll
        for (int p = 0; p < PT; ++p) {
          floatx4 x;
#pragma unroll
          for (int r = 0; r < 4; ++r) x[r] = xs[(16 * jb + 4 * grp + r) * LX + 16 * p + fr];
          u[p] += mfma16(b, x, floatx4{0.f, 0.f, 0.f, 0.f});
        }
      }
#pragma unroll
      for (int p = 0; p < PT; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[k][p][r] = __builtin_fmaf(S[k][p][r], dec, u[p][r]);
    }
  }
#pragma unroll
  for (int k = 0; k < NW; ++k)
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
      for (int r = 0; r < 4; ++r) sp[(size_t)(16 * (NW * w + k) + 4 * grp + r) * a.P + 16 * p + fr] = S[k][p][r];
}

}  // namespace

extern "C" int fls_seq_ssd_scan_chunked(const float* xbc, int ldx, const float* z, int ldz, const float* dt, int lddt, const float* dt_bias,
                                        const float* A_log, const float* Dskip, float* state, float* out, int ldo, const int* cu,
                                        const int* pos0, const int* slot, int B, int max_rows, int nh, int P, int N, int G, float* scratch,
                                        fls_stream_t s) {
  if (B <= 0 || max_rows <= 0) return 0;
  // rows of four: B, C and x are read 16 bytes at a time
  if ((N != 64 && N != 128) || P % 16 || G < 1 || nh % G || ldx % 4 || (uintptr_t)xbc % 16 || scratch == nullptr || (uintptr_t)scratch % 16) return -1;
  const Ssd a = {xbc, ldx, z, ldz, dt, lddt, dt_bias, A_log, Dskip, state, out, ldo, cu, pos0, slot, nh, P, N, G, scratch};
  const hipStream_t st = (hipStream_t)s;
  const dim3 chunks((max_rows + CQ - 1) / CQ, G, B);
  if (N == 128) hipLaunchKernelGGL(ssd_scores_kernel<128>, chunks, dim3(256), 0, st, a);
  else hipLaunchKernelGGL(ssd_scores_kernel<64>, chunks, dim3(256), 0, st, a);
  SEQ_LAUNCH_CHECK();
  // two column tiles a block read B and C half as often; one where that would leave CUs without a block
  const bool two = P % 32 == 0 && (long long)B * nh * (P / 32) >= 256;
#define SSD(PT, NW) hipLaunchKernelGGL((ssd_chunk_kernel<PT, NW>), dim3(P / (16 * PT), nh, B), dim3(256), 0, st, a)
  if (N == 128) { if (two) SSD(2, 2); else SSD(1, 2); }
  else { if (two) SSD(2, 1); else SSD(1, 1); }
#undef SSD
  SEQ_LAUNCH_CHECK();
  return 0;
}
