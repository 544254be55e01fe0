// Prompt attention on the matrix cores, for bf16 models: the same masks (chunk, window, kept first
// keys), score cap, distance penalty and weights (softmax, or a sigmoid gate per key) as
// attn_paged_kernel, for steps that bring many rows per request.  Queries may come as fp32 (rounded to
// bf16 on their way into the fragments).  Keys of a row tile: first the kept first keys that lie before
// the tile's window (if any), then the window's keys, both walked 32 at a time.
//
// POOL (beside a window): ahead of the window's tiles come tiles of block means, one key and value for each block of
// ab.P positions that ends before the window, from block pools with pages of their own; query i sees blocks
// b < (i - window + 1) / ab.P.
//
// The host cuts every request's rows of the step into tiles of up to 128 consecutive rows; a block
// serves one tile and one query head, its four waves 32 query rows each.  Keys are walked 64 at a
// time, from the first key the tile's first row may see to the tile's last row, gathered from the
// request's pages into LDS: K as [key][d], V transposed as [column][key].  Per half of a key tile and wave:
//   S^T = K Q^T        one 32x32x16 MFMA per 16 of d (Q fragments stay in registers): a lane then
//                      holds 16 keys' scores of ONE query (column = lane % 32), its partner lane ^ 32
//                      the other 16, so the softmax statistics are per-lane scalars: one shuffle
//                      per reduction, and the running maximum, sum and rescale factor live in the
//                      lane that owns the query;
//   scores             scale, cap, distance penalty, mask (chunk / window / causal) in fp32;
//   weights            exp in fp32, then two bf16 terms (p = hi + lo, 16 mantissa bits together), so the
//                      value product loses nothing to a bf16 rounding of p;
//   O^T += V^T P^T     MFMAs again; O^T has the same column = query layout, so the rescale is a
//                      per-lane multiply.  The keys of V's rows stand in the order in which a lane holds
//                      its scores, so the weights are the operand as they are.
//
// What bounds it is the vector work per score beside the matrix work (24 MFMAs, 768 cycles, per half tile and wave with heads of
// 128), with two waves a SIMD to overlap them.  So scores are in units of log 2: exp and log are one instruction each and the penalty
// needs no factor.  The cap and the sigmoid weights come from exp(-|x|) and a reciprocal of [1, 2] that one Newton step makes as exact
// as a division.  bf16 terms come from the conversion instruction, and a half tile that every row of the wave sees has no mask.  The
// accumulators are rescaled when a maximum grows, and only then: a query's largest weight is exactly 1, which two bf16 terms hold without
// error (left up to 2^8 behind the maximum, outputs were up to twice as far from 64 bits, for 4% of the time).  A half tile has 63
// different distances: a lane works out the penalty of one and reads its 16 from LDS.  The pool row of every key is found once, a tile
// ahead, by one thread (every 16-byte piece used to look its page up, 12 a thread and tile).  Weights pass to the value product in
// registers (through LDS before), maxima cross lanes without LDS, sums meet at the end, and a kernel for each kind of weight
// leaves no branch in a score's way.  All heads of a group run on one XCD, whose L2 then holds the group's keys once (fetched from
// memory, 8 prompts of 2048 with 32 heads on 8: 250 MB -> 105).  Before and after these:
//   8 of 2048, 32 heads of 128 on 8, cap and penalty   988 -> 663 us      4 of 1500, 48 on 8, plain             379 -> 230 us
//   9 of 510 .. 1501, 16 on 16, plain, fp32 queries    250 -> 140         the same with a window of 1024        221 -> 129
//   6 of 610 .. 1800, 16 on 4, sigmoid, window 512     137 -> 92          2 x 512 rows at 512, 16 on 4, penalty 88 -> 60
//   6 of 1500, 16 heads of 64 on 4, cap and penalty    195 -> 135         3 of 37 .. 120                        17.3 -> 14.0
// (both halves of a tile at once spill: 718 us in the first, 136 in the windowed one.)
#include "seq_common.h"
#include "fls_seq.h"

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

#define KT 32             // keys per tile
#define PLD (KT + 8)      // row stride (elements) of the transposed V tile of 32 keys
#define PT 64             // keys per tile of the prompt kernel, worked on in halves of KT
#define VLD (PT + 8)
#define LOG2E 1.4426950408889634f

__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float log2_hw(float x) { return __builtin_amdgcn_logf(x); }
// 1 / x for x in [1, 2], as a division rounds it: the hardware's reciprocal and one Newton step
__device__ __forceinline__ float rcp_near(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.f), r, r);
}

// maximum / sum over lanes l and l ^ 32, in both
__device__ __forceinline__ float halves_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// eight weights as two bf16 terms each
__device__ __forceinline__ void two_terms(const float* p, bf16x8& hi, bf16x8& lo) {
  typedef float floatx8 __attribute__((ext_vector_type(8)));
  floatx8 v;
#pragma unroll
  for (int x = 0; x < 8; ++x) v[x] = p[x];
  hi = __builtin_convertvector(v, bf16x8);
  lo = __builtin_convertvector(v - __builtin_convertvector(hi, floatx8), bf16x8);
}

// (two waves per SIMD: a few registers over 256 would halve that)
// KIND: 0 softmax of the scaled scores, 1 with a cap and / or a distance penalty, 2 sigmoid weights
template <int D, int DV, typename TQ, typename TO, bool POOL, int KIND>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(const TQ* __restrict__ q, int ldq, const bf16_t* __restrict__ kc, int ldk,
                                                           const bf16_t* __restrict__ vc, int ldv, TO* __restrict__ out, int ldo,
                                                           const int* __restrict__ tiles, const int* __restrict__ tok_seq,
                                                           const int* __restrict__ tok_pos, const int* __restrict__ page_table,
                                                           int pt_stride, int H, int G, float scale, float softcap,
                                                           const float* __restrict__ r1, const float* __restrict__ r2,
                                                           int chunk, int window, int keep_first,
                                                           const float* __restrict__ gate_bias, float out_scale, int page_size,
                                                           int has_sink, float sink, const float* __restrict__ sink_h,
                                                           const float* __restrict__ head_gate,
                                                           int ldhg, int Gv, AttnBlocks ab, int page_shift) {
  constexpr int KLD = D + 8;
  __shared__ __attribute__((aligned(16))) bf16_t Ks[PT * KLD];
  __shared__ __attribute__((aligned(16))) bf16_t Vt[DV * VLD];
  __shared__ __attribute__((aligned(8))) int rows[PT];               // pool rows of the tile that is fetched next
  __shared__ float pen[4][64];                                       // a wave's distance penalties of a half tile
  // (blocks go to the XCDs in turn: a group's heads onto one of them)
  const int h = H % 8 ? (int)blockIdx.x : (int)(blockIdx.x % 8) * (H / 8) + (int)blockIdx.x / 8, g = h / (H / G);
  const int tile = gridDim.y - 1 - blockIdx.y;                       // (the last tiles of a long prompt have the most keys: they go first)
  const int row0 = tiles[2 * tile], nrows = tiles[2 * tile + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ql = lane & 31, h2 = lane >> 5;
  const int* table = page_table + (size_t)tok_seq[row0] * pt_stride;
  const int i_first = tok_pos[row0], i_last = i_first + nrows - 1;
  // this lane's query
  const int qrow = wave * 32 + ql;
  const bool qok = qrow < nrows;
  const int iq = i_first + qrow;
  int lo_q = chunk > 0 ? (iq / chunk) * chunk : 0;
  if (window > 0 && iq - window + 1 > lo_q) lo_q = iq - window + 1;
  int lo_blk = chunk > 0 ? (i_first / chunk) * chunk : 0;
  if (window > 0 && i_first - window + 1 > lo_blk) lo_blk = i_first - window + 1;
  // the wave's rows span positions [w_first, w_last]; it skips key tiles none of them sees
  const int w_first = i_first + wave * 32, w_last = min(i_last, w_first + 31);
  int lo_w = chunk > 0 ? (w_first / chunk) * chunk : 0;
  if (window > 0 && w_first - window + 1 > lo_w) lo_w = w_first - window + 1;
  int lo_wl = chunk > 0 ? (w_last / chunk) * chunk : 0;              // the first key that the wave's last row sees: the latest of its rows
  if (window > 0 && w_last - window + 1 > lo_wl) lo_wl = w_last - window + 1;
  bf16x8 Qf[D / 16];
  {
    const TQ* qp = q + (size_t)(row0 + (qok ? qrow : 0)) * ldq + (size_t)h * D + h2 * 8;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (qok) {
        if constexpr (sizeof(TQ) == 2) {
          v = *reinterpret_cast<const uint4*>(qp + 16 * s);
        } else {
          const float4 f0 = *reinterpret_cast<const float4*>(qp + 16 * s), f1 = *reinterpret_cast<const float4*>(qp + 16 * s + 4);
          bf16_t e[8] = {f_to_bf16(f0.x), f_to_bf16(f0.y), f_to_bf16(f0.z), f_to_bf16(f0.w),
                         f_to_bf16(f1.x), f_to_bf16(f1.y), f_to_bf16(f1.z), f_to_bf16(f1.w)};
          v = *reinterpret_cast<const uint4*>(e);
        }
      }
      Qf[s] = *reinterpret_cast<bf16x8*>(&v);
    }
  }
  floatx16 O[DV / 32];
#pragma unroll
  for (int c = 0; c < DV / 32; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) O[c][r] = 0.f;
  // (the softmax's silent entry of score `sink` / sink_h[h], if any, is where every query's running maximum and sum start)
  // (a lane sums its own keys: the two sums of a query meet at the end)
  float m = has_sink ? (sink_h != nullptr ? sink_h[h] : sink) * LOG2E : -1e30f, l = has_sink && h2 == 0 ? 1.f : 0.f;
  const float a1 = r1 != nullptr ? r1[h] : 0.f, a2 = r2 != nullptr ? r2[h] : 0.f;
  constexpr bool gated = KIND == 2;
  const float gb = gated ? gate_bias[h] * LOG2E : 0.f;
  // scores in units of log 2; with a cap: cap (1 - 2 / (exp(2 s / cap) + 1)), the exponential's argument straight from the product
  const float sc_mul = softcap > 0.f ? 2.f * LOG2E * scale / softcap : scale * LOG2E;
  const float cap2 = softcap * LOG2E;
  // key tiles: nt_keep tiles over the kept first keys [0, nkeep) that lie before the block's window,
  // then the tiles from lo_blk to the block's last row
  // (POOL: instead nt_keep tiles over the blocks [0, nkeep) that the block's last row sees)
  auto seen_blocks = [&](int i) { return i - window + 1 > 0 ? (i - window + 1) / ab.P : 0; };
  const int nkeep = POOL ? seen_blocks(i_last) : min(keep_first, lo_blk);
  const int keep_q = POOL ? seen_blocks(iq) : keep_first;            // what of them this lane's query sees ...
  const int keep_w = POOL ? seen_blocks(w_last) : keep_first;        // ... and any of the wave's
  const int* btable = POOL ? ab.table + (size_t)tok_seq[row0] * ab.t_stride : nullptr;
  const int nt_keep = (nkeep + PT - 1) / PT;
  const int nt = nt_keep + (i_last - lo_blk) / PT + 1;
  // K / V of a key tile travel global -> registers -> LDS; the next tile's loads are issued before this
  // tile's matrix work and land in LDS after it, so the page gather's latency hides under the MFMAs
  constexpr int PK = PT * (D / 8), PV = PT / 2 * (DV / 8);           // 16-byte pieces of K; pieces of two neighbouring keys of V
  constexpr int NK = (PK + 255) / 256, NV = (PV + 255) / 256;        // per thread (the last one of some threads may be none)
  u32x4 kreg[NK], vreg[NV][2];
  // rows of the pools that hold a tile's keys: one thread a key, kept in LDS a tile ahead of the loads that use them (keys behind
  // the tile's last are that one again: every row masks them)
  auto find_row = [&](int ti) {
    const bool pre = ti < nt_keep;
    const int j0 = pre ? ti * PT : lo_blk + (ti - nt_keep) * PT;
    const int j = min(j0 + (int)threadIdx.x, (pre ? nkeep : i_last + 1) - 1);
    const int* tab = POOL && pre ? btable : table;
    const int pg = page_shift >= 0 ? j >> page_shift : j / page_size;
    return int2{tab[pg], j - pg * page_size};
  };
  const int vpair = threadIdx.x % (PT / 2);
  auto fetch = [&](int ti) {
    const bool pre = POOL && ti < nt_keep;
    const bf16_t* kb = pre ? reinterpret_cast<const bf16_t*>(ab.kp) : kc;
    const bf16_t* vb = pre ? reinterpret_cast<const bf16_t*>(ab.vp) : vc;
    const int lk = pre ? ab.ldk : ldk, lv = pre ? ab.ldv : ldv;
    kb += (size_t)g * D;
    vb += (size_t)(g % Gv) * DV;
#pragma unroll
    for (int x = 0; x < NK; ++x) {
      const int e = threadIdx.x + 256 * x;
      if (PK % 256 == 0 || e < PK) kreg[x] = *reinterpret_cast<const u32x4*>(kb + (size_t)rows[e / (D / 8)] * lk + e % (D / 8) * 8);
    }
    const int2 vr = *reinterpret_cast<const int2*>(rows + 2 * vpair);
    const bf16_t* v0 = vb + (size_t)vr.x * lv;
    const bf16_t* v1 = vb + (size_t)vr.y * lv;
#pragma unroll
    for (int x = 0; x < NV; ++x) {
      const int e = threadIdx.x + 256 * x;
      if (PV % 256 == 0 || e < PV) {
        vreg[x][0] = *reinterpret_cast<const u32x4*>(v0 + e / (PT / 2) * 8);
        vreg[x][1] = *reinterpret_cast<const u32x4*>(v1 + e / (PT / 2) * 8);
      }
    }
  };
  // (a key's place in a row of the transposed V: keys 4 .. 7 and 8 .. 11 of every 16 change places, so that the weights a lane
  // holds are the values' operand as they stand)
  const int vplace = (vpair & ~6) | (vpair & 2) << 1 | (vpair & 4) >> 1;
  int2 next_row = {0, 0};
  if (threadIdx.x < PT) {
    const int2 r = find_row(0);
    rows[threadIdx.x] = r.x * page_size + r.y;
    if (nt > 1) next_row = find_row(1);
  }
  __syncthreads();
  fetch(0);
  for (int ti = 0; ti < nt; ++ti) {
    const bool kept = ti < nt_keep;
    const int jt = kept ? ti * PT : lo_blk + (ti - nt_keep) * PT;
    const int jend = kept ? nkeep : i_last + 1;      // keys from jend on are padding of this tile
    __syncthreads();                          // the previous tile's readers are done
    if (threadIdx.x < PT) rows[threadIdx.x] = next_row.x * page_size + next_row.y;
#pragma unroll
    for (int x = 0; x < NK; ++x) {
      const int e = threadIdx.x + 256 * x;
      if (PK % 256 == 0 || e < PK) *reinterpret_cast<u32x4*>(Ks + (e / (D / 8)) * KLD + (e % (D / 8)) * 8) = kreg[x];
    }
#pragma unroll
    for (int x = 0; x < NV; ++x) {            // (two keys of a column make one 4-byte store)
      const int e = threadIdx.x + 256 * x;
      if (PV % 256 != 0 && e >= PV) continue;
      uint32_t* dst = reinterpret_cast<uint32_t*>(Vt + (e / (PT / 2)) * 8 * VLD) + vplace;
      const uint32_t a[4] = {vreg[x][0].x, vreg[x][0].y, vreg[x][0].z, vreg[x][0].w}, b[4] = {vreg[x][1].x, vreg[x][1].y, vreg[x][1].z, vreg[x][1].w};
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        dst[2 * y * (VLD / 2)] = __builtin_amdgcn_perm(b[y], a[y], 0x05040100);
        dst[(2 * y + 1) * (VLD / 2)] = __builtin_amdgcn_perm(b[y], a[y], 0x07060302);
      }
    }
    __syncthreads();
    if (ti + 1 < nt) fetch(ti + 1);
    if (ti + 2 < nt && threadIdx.x < PT) next_row = find_row(ti + 2);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
    const int j0 = jt + half * KT;
    if (j0 >= jend || wave * 32 >= nrows || (POOL && kept && j0 >= keep_w) ||
        (!kept && (j0 > w_last || (j0 + KT - 1 < lo_w && (POOL || j0 >= keep_first))))) continue;   // (wave-uniform)
    // every row of the wave sees every key of this half (rows past the tile's end compute what nobody stores)
    const bool full = !kept && j0 + KT - 1 <= w_first && j0 >= lo_wl;
    // a distance penalty depends on query - key alone, 63 of them a half tile: a lane works out one
    if (KIND != 0 && a1 != 0.f) pen[wave][lane] = log2_hw(1.f + a2 * fmaxf((float)(w_first - j0 + 31 - lane), 0.f));
    floatx16 S;
#pragma unroll
    for (int r = 0; r < 16; ++r) S[r] = 0.f;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
      const bf16x8 kf = *reinterpret_cast<const bf16x8*>(Ks + (half * KT + ql) * KLD + 16 * s + h2 * 8);
      S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, Qf[s], S, 0, 0, 0);
    }
    float p[16];
    float mt = -1e30f;
    // (this kernel serves bf16 models only: the hardware exp / log are far inside their rounding)
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = S[r] * sc_mul;
    if (KIND != 0 && softcap > 0.f) {          // cap tanh: (1 - e) / (1 + e), e = exp(-2 |s| / cap), never overflows or cancels
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float e = exp2_hw(-fabsf(p[r]));
        p[r] = copysignf(__builtin_fmaf(-cap2, e, cap2) * rcp_near(1.f + e), p[r]);
      }
    }
    if (KIND != 0 && a1 != 0.f) {
      // (other lanes' entries: LDS is in order per wave, but the compiler must neither move these loads above the stores nor the next
      // half's stores above these loads)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const float* pq = pen[wave] + 31 - ql + 4 * h2;
#pragma unroll
      for (int r = 0; r < 16; ++r) p[r] -= a1 * pq[8 * (r >> 2) + (r & 3)];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    if (gated) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float y = p[r] + gb, e = exp2_hw(-fabsf(y)), q = rcp_near(1.f + e);
        p[r] = y < 0.f ? e * q : q;
      }
    }
    if (!full) {
      // the row sees keys [mlo, mhi] and, of a window's tiles, those before keep_first (no key of a row past the tile's end)
      const int jb = j0 + 4 * h2;
      const int mlo = (kept ? 0 : lo_q) - jb, mkeep = (POOL ? 0 : keep_first) - jb;
      const int mhi = (!qok ? -1 : POOL ? (kept ? keep_q - 1 : iq) : min(iq, jend - 1)) - jb;
      const float hidden = gated ? 0.f : -1e30f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int o = 8 * (r >> 2) + (r & 3);
        const bool vis = (o <= mhi) & ((o >= mlo) | (o < mkeep));
        p[r] = vis ? p[r] : hidden;
      }
    }
    if (!gated) {
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, p[r]);
      mt = halves_max(mt);
      if (__any(mt > m)) {               // (wave-uniform)
        mt = fmaxf(mt, m);
        const float corr = exp2_hw(m - mt);
        l *= corr;
        m = mt;
#pragma unroll
        for (int c = 0; c < DV / 32; ++c)
#pragma unroll
          for (int r = 0; r < 16; ++r) O[c][r] *= corr;
      }
      float ps = 0.f;
      if (full) {
#pragma unroll
        for (int r = 0; r < 16; ++r) { p[r] = exp2_hw(p[r] - m); ps += p[r]; }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) { p[r] = p[r] > -1e29f ? exp2_hw(p[r] - m) : 0.f; ps += p[r]; }
      }
      l += ps;
    }
    // two bf16 terms of each weight, in the order of the keys of a row of V
    bf16x8 ph[KT / 16], pl[KT / 16];
#pragma unroll
    for (int ks = 0; ks < KT / 16; ++ks) two_terms(p + 8 * ks, ph[ks], pl[ks]);
#pragma unroll
    for (int ks = 0; ks < KT / 16; ++ks) {
#pragma unroll
      for (int c = 0; c < DV / 32; ++c) {
        const bf16x8 vf = *reinterpret_cast<const bf16x8*>(Vt + (32 * c + ql) * VLD + half * KT + 16 * ks + 8 * h2);
        O[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, ph[ks], O[c], 0, 0, 0);
        O[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pl[ks], O[c], 0, 0, 0);
      }
    }
    }
  }
  l = halves_sum(l);
  if (qok && (gated || l > 0.f)) {
    float inv = gated ? out_scale : out_scale / l;
    if (head_gate != nullptr) inv *= sigmoid_f(head_gate[(size_t)(row0 + qrow) * ldhg + h]);
    TO* op = out + (size_t)(row0 + qrow) * ldo + (size_t)h * DV;
#pragma unroll
    for (int c = 0; c < DV / 32; ++c)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        if constexpr (sizeof(TO) == 4) {
          *reinterpret_cast<float4*>(op + 32 * c + 8 * rg + 4 * h2) =
              make_float4(O[c][4 * rg] * inv, O[c][4 * rg + 1] * inv, O[c][4 * rg + 2] * inv, O[c][4 * rg + 3] * inv);
        } else {
          bf16_t o4[4];
#pragma unroll
          for (int x = 0; x < 4; ++x) o4[x] = f_to_bf16(O[c][4 * rg + x] * inv);
          *reinterpret_cast<uint2*>(op + 32 * c + 8 * rg + 4 * h2) = *reinterpret_cast<const uint2*>(o4);
        }
      }
  }
}

// tiles: n_tiles x (first packed row, rows <= 128) of one request each.  tq: type of q (0 fp32, 1 bf16);
// pools are bf16, out of type to.  Gv (0: G): value heads in the pool, key head g reads value head g % Gv.  Returns -2 for head sizes or alignments this kernel does not serve (the
// caller then runs fls_seq_attn_paged).
extern "C" int fls_seq_attn_prefill(const void* q, int ldq, int tq, const void* kc, int ldk, const void* vc, int ldv, void* out,
                                    int to, int ldo, const int* tiles, int n_tiles, const int* tok_seq, const int* tok_pos,
                                    const int* page_table, int pt_stride, int H, int G, int d, int dv, float scale,
                                    float softcap, const float* r1, const float* r2, int chunk, int window, int keep_first,
                                    const float* gate_bias, float out_scale, int page_size, int has_sink, float sink, const float* sink_h,
                                    const float* head_gate, int ldhg, int Gv, int pool_P, const void* kp, int ldkp, const void* vp,
                                    int ldvp, const int* block_table, int bt_stride, fls_stream_t s) {
  if (n_tiles <= 0) return 0;
  if (has_sink && gate_bias != nullptr) return -1;
  if (Gv <= 0) Gv = G;
  if (G < 1 || H % G || G % Gv || page_size < 1 || ldq % 8 || ldo % 4 || ldk % 8 || ldv % 8 || G * d > ldk || Gv * dv > ldv ||
      (uintptr_t)q % 16 || (uintptr_t)kc % 16 || (uintptr_t)vc % 16 || (uintptr_t)out % 16 || keep_first < 0)
    return -2;
  if (pool_P < 0 || (pool_P > 0 && (window < 1 || chunk > 0 || keep_first > 0 || has_sink || gate_bias != nullptr || r1 != nullptr ||
                                    kp == nullptr || vp == nullptr || block_table == nullptr || G * d > ldkp || Gv * dv > ldvp)))
    return -1;                                          // (blocks go with a plain softmax over a window)
  if (pool_P > 0 && (tq != 0 || ldkp % 8 || ldvp % 8 || (uintptr_t)kp % 16 || (uintptr_t)vp % 16)) return -2;
  const AttnBlocks ab = {pool_P, kp, ldkp, vp, ldvp, block_table, bt_stride};
  const int page_shift = (page_size & (page_size - 1)) == 0 ? __builtin_ctz(page_size) : -1;
  dim3 grid(H, n_tiles);
  hipStream_t st = (hipStream_t)s;
#define ATTN_PF_(DD, DDV, TQ_, TO_, PP, KK)                                                                                   \
  hipLaunchKernelGGL((attn_prefill_kernel<DD, DDV, TQ_, TO_, PP, KK>), grid, dim3(256), 0, st, (const TQ_*)q, ldq,            \
                     (const bf16_t*)kc, ldk, (const bf16_t*)vc, ldv, (TO_*)out, ldo, tiles, tok_seq, tok_pos,             \
                     page_table, pt_stride, H, G, scale, softcap, r1, r2, chunk, window, keep_first, gate_bias,           \
                     out_scale, page_size, has_sink, sink, sink_h, head_gate, ldhg, Gv, ab, page_shift)
#define ATTN_PF_KIND(DD, DDV, TQ_, TO_)                                                                                   \
  do {                                                                                                                    \
    if (gate_bias != nullptr) ATTN_PF_(DD, DDV, TQ_, TO_, false, 2);                                                      \
    else if (softcap > 0.f || r1 != nullptr) ATTN_PF_(DD, DDV, TQ_, TO_, false, 1);                                       \
    else ATTN_PF_(DD, DDV, TQ_, TO_, false, 0);                                                                           \
  } while (0)
#define ATTN_PF(DD, DDV)                                                                                                  \
  do {                                                                                                                    \
    if (tq == 1 && to == 1) ATTN_PF_KIND(DD, DDV, bf16_t, bf16_t);                                                        \
    else if (tq == 1) ATTN_PF_KIND(DD, DDV, bf16_t, float);                                                               \
    else if (to == 1) ATTN_PF_KIND(DD, DDV, float, bf16_t);                                                               \
    else ATTN_PF_KIND(DD, DDV, float, float);                                                                             \
  } while (0)
#define ATTN_PF_POOL(DD, DDV)                                                                                             \
  do {                                                                                                                    \
    if (softcap > 0.f) {                                                                                                  \
      if (to == 1) ATTN_PF_(DD, DDV, float, bf16_t, true, 1);                                                             \
      else ATTN_PF_(DD, DDV, float, float, true, 1);                                                                      \
    } else if (to == 1) ATTN_PF_(DD, DDV, float, bf16_t, true, 0);                                                        \
    else ATTN_PF_(DD, DDV, float, float, true, 0);                                                                        \
  } while (0)
  if (pool_P > 0) {
    if (d == 128 && dv == 128) ATTN_PF_POOL(128, 128);
    else if (d == 96 && dv == 96) ATTN_PF_POOL(96, 96);
    else if (d == 64 && dv == 64) ATTN_PF_POOL(64, 64);
    else if (d == 32 && dv == 32) ATTN_PF_POOL(32, 32);
    else if (d == 128 && dv == 64) ATTN_PF_POOL(128, 64);
    else if (d == 64 && dv == 128) ATTN_PF_POOL(64, 128);
    else return -2;
  } else if (d == 128 && dv == 128) ATTN_PF(128, 128);
  else if (d == 64 && dv == 64) ATTN_PF(64, 64);
  else if (d == 128 && dv == 64) ATTN_PF(128, 64);
  else if (d == 64 && dv == 128) ATTN_PF(64, 128);
  else return -2;
#undef ATTN_PF_POOL
#undef ATTN_PF
#undef ATTN_PF_KIND
#undef ATTN_PF_
  SEQ_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------- few rows, many heads on one key/value head
// Decode rows of an attention whose query heads share one key / value head -- attention over cached latent
// rows: every head reads the same long rows (keys D wide, values their first DV columns or a pool of their
// own).  Here the HEADS of one token are the 32 query columns of the MFMA tile: a block serves (token,
// key/value head, range of key tiles), stages each tile of 32 rows once in LDS for all heads, and its four
// waves share the score product's operands but own a quarter of the value columns each, so every wave
// keeps DV / 4 accumulator columns.  All waves compute the same scores and softmax statistics (no exchange
// between them) and pass the weights on in registers, as above.  A block whose range is one of several
// leaves (maximum, sum, weighted values) in `part` for attn_merge_kernel.  A block mostly walks a tile or two, so what bounds it is
// the chain up to its first product and the code it fetches for it: keys' rows are found by a thread a key (each 16-byte piece divided
// by the page size and read the table before), queries past the last head are not laid down, two keys of V make one store.  Merge
// included, 24 tokens of 16 heads on rows of 576, 130 keys in 8 ranges 22.0 -> 15.2 us; of 512, 1,024 keys 44.6 -> 25.5; 5 of 256,
// 90 keys in one 16.0 -> 9.3.
template <int D, int DV>
__global__ __launch_bounds__(256) void attn_heads_kernel(const float* __restrict__ q, int ldq, const bf16_t* kc, int ldk,
                                                         const bf16_t* vc, int ldv, bf16_t* __restrict__ out, int ldo,
                                                         const int* __restrict__ tok_seq, const int* __restrict__ tok_pos,
                                                         const int* __restrict__ page_table, int pt_stride, int H, int G,
                                                         float scale, int window, int keep_first, float out_scale,
                                                         int page_size, float* __restrict__ part, const float* __restrict__ sink_h,
                                                         const float* __restrict__ head_gate, int ldhg, int page_shift) {
  constexpr int KLD = D + 8;
  constexpr int CPW = DV / 128;               // 32-column blocks of the values per wave
  __shared__ __attribute__((aligned(16))) bf16_t Ks[KT * KLD];
  __shared__ __attribute__((aligned(16))) bf16_t Vt[DV * PLD];
  __shared__ __attribute__((aligned(8))) int rows[KT];               // pool rows of the tile that is fetched next
  const int t = blockIdx.x, g = blockIdx.y, nsplit = gridDim.z;
  const int nh = H / G;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ql = lane & 31, h2 = lane >> 5;
  const int* table = page_table + (size_t)tok_seq[t] * pt_stride;
  const int i = tok_pos[t];
  const int lo = window > 0 ? max(0, i - window + 1) : 0;
  const int nkeep = min(keep_first, lo);
  const int nt_keep = (nkeep + KT - 1) / KT;
  const int nt = nt_keep + (i - lo) / KT + 1;
  const int tps = (nt + nsplit - 1) / nsplit;
  const int ti_lo = blockIdx.z * tps, ti_hi = min(nt, ti_lo + tps);
  const bool qok = ql < nh;
  const int head = g * nh + (qok ? ql : 0);
  // rows of the pools that hold a tile's keys, one thread a key (keys behind the tile's last are that one again, and masked)
  auto find_row = [&](int ti) {
    const bool kept = ti < nt_keep;
    const int j0 = kept ? ti * KT : lo + (ti - nt_keep) * KT;
    const int j = min(j0 + (int)threadIdx.x, (kept ? nkeep : i + 1) - 1);
    const int pg = page_shift >= 0 ? j >> page_shift : j / page_size;
    return int2{table[pg], j - pg * page_size};
  };
  const bool any = ti_lo < ti_hi;
  int2 next_row = {0, 0};
  if (any && threadIdx.x < KT) next_row = find_row(ti_lo);
  // the token's queries: read once by the whole block (16-byte loads over the heads' contiguous rows),
  // rounded to bf16 into the key tile's LDS, and from there into every wave's fragments (what stands there for heads past the last
  // makes scores that are masked)
  bf16x8 Qf[D / 16];
  {
    const float* qb = q + (size_t)t * ldq + (size_t)g * nh * D;
#pragma unroll 3
    for (int e = threadIdx.x; e < (any ? nh * (D / 4) : 0); e += 256) {
      const int hh = e / (D / 4), c4 = e % (D / 4);
      const floatx4 f = *reinterpret_cast<const floatx4*>(qb + (size_t)hh * D + c4 * 4);
      *reinterpret_cast<bf16x4*>(Ks + hh * KLD + c4 * 4) = __builtin_convertvector(f, bf16x4);
    }
    if (any && threadIdx.x < KT) rows[threadIdx.x] = next_row.x * page_size + next_row.y;
    __syncthreads();
#pragma unroll
    for (int s = 0; s < D / 16; ++s) Qf[s] = *reinterpret_cast<const bf16x8*>(Ks + ql * KLD + 16 * s + h2 * 8);
  }
  floatx16 O[CPW];
#pragma unroll
  for (int c = 0; c < CPW; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) O[c][r] = 0.f;
  // (a silent softmax entry of score sink_h[head] is where the running maximum and sum start; with ranges the merge adds it)
  const bool snk = sink_h != nullptr && nsplit == 1;
  float m = snk ? sink_h[head] : -1e30f, l = snk ? 1.f : 0.f;
  constexpr int NK = KT * (D / 8) / 256, NV = KT / 2 * (DV / 8) / 256;       // pieces of K; pieces of two neighbouring keys of V
  static_assert(NK >= 1 && NV >= 1 && KT * (D / 8) % 256 == 0 && KT / 2 * (DV / 8) % 256 == 0 && CPW >= 1, "tile pieces per thread");
  const int vpair = threadIdx.x % (KT / 2);
  const int vplace = (vpair & ~6) | (vpair & 2) << 1 | (vpair & 4) >> 1;     // (as in the prompt kernel)
  u32x4 kreg[NK], vreg[NV][2];
  auto fetch = [&]() {
    const bf16_t* kb = kc + (size_t)g * D;
#pragma unroll
    for (int x = 0; x < NK; ++x) {
      const int e = threadIdx.x + 256 * x;
      kreg[x] = *reinterpret_cast<const u32x4*>(kb + (size_t)rows[e / (D / 8)] * ldk + e % (D / 8) * 8);
    }
    const int2 vr = *reinterpret_cast<const int2*>(rows + 2 * vpair);
    const bf16_t* v0 = vc + (size_t)vr.x * ldv + (size_t)g * DV;
    const bf16_t* v1 = vc + (size_t)vr.y * ldv + (size_t)g * DV;
#pragma unroll
    for (int x = 0; x < NV; ++x) {
      const int seg = (threadIdx.x + 256 * x) / (KT / 2);
      vreg[x][0] = *reinterpret_cast<const u32x4*>(v0 + seg * 8);
      vreg[x][1] = *reinterpret_cast<const u32x4*>(v1 + seg * 8);
    }
  };
  if (any) fetch();
  if (ti_lo + 1 < ti_hi && threadIdx.x < KT) next_row = find_row(ti_lo + 1);
  for (int ti = ti_lo; ti < ti_hi; ++ti) {
    const bool kept = ti < nt_keep;
    const int j0 = kept ? ti * KT : lo + (ti - nt_keep) * KT;
    const int jend = kept ? nkeep : i + 1;
    __syncthreads();
    if (threadIdx.x < KT) rows[threadIdx.x] = next_row.x * page_size + next_row.y;
#pragma unroll
    for (int x = 0; x < NK; ++x) {
      const int e = threadIdx.x + 256 * x;
      *reinterpret_cast<u32x4*>(Ks + (e / (D / 8)) * KLD + (e % (D / 8)) * 8) = kreg[x];
    }
#pragma unroll
    for (int x = 0; x < NV; ++x) {
      uint32_t* dst = reinterpret_cast<uint32_t*>(Vt + (threadIdx.x + 256 * x) / (KT / 2) * 8 * PLD) + vplace;
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        dst[2 * y * (PLD / 2)] = __builtin_amdgcn_perm(vreg[x][1][y], vreg[x][0][y], 0x05040100);
        dst[(2 * y + 1) * (PLD / 2)] = __builtin_amdgcn_perm(vreg[x][1][y], vreg[x][0][y], 0x07060302);
      }
    }
    __syncthreads();
    if (ti + 1 < ti_hi) fetch();
    if (ti + 2 < ti_hi && threadIdx.x < KT) next_row = find_row(ti + 2);
    floatx16 S;
#pragma unroll
    for (int r = 0; r < 16; ++r) S[r] = 0.f;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
      const bf16x8 kf = *reinterpret_cast<const bf16x8*>(Ks + ql * KLD + 16 * s + h2 * 8);
      S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, Qf[s], S, 0, 0, 0);
    }
    float p[16];
    float mt = -1e30f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int j = j0 + 8 * (r >> 2) + 4 * h2 + (r & 3);
      const bool vis = qok && j < jend;            // (every key of a tile below jend is visible: j <= i, inside the window or kept)
      p[r] = vis ? S[r] * scale : -1e30f;
      mt = fmaxf(mt, p[r]);
    }
    mt = fmaxf(halves_max(mt), m);
    float ps = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      p[r] = p[r] > -1e29f ? __expf(p[r] - mt) : 0.f;
      ps += p[r];
    }
    ps = halves_sum(ps);
    const float corr = __expf(m - mt);
    l = l * corr + ps;
    m = mt;
#pragma unroll
    for (int c = 0; c < CPW; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) O[c][r] *= corr;
#pragma unroll
    for (int ks = 0; ks < KT / 16; ++ks) {
      bf16x8 ph, pl;
      two_terms(p + 8 * ks, ph, pl);
#pragma unroll
      for (int c = 0; c < CPW; ++c) {
        const bf16x8 vf = *reinterpret_cast<const bf16x8*>(Vt + (32 * (wave * CPW + c) + ql) * PLD + 16 * ks + 8 * h2);
        O[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, ph, O[c], 0, 0, 0);
        O[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pl, O[c], 0, 0, 0);
      }
    }
  }
  if (!qok) return;
  if (nsplit == 1) {
    float inv = out_scale / l;
    if (head_gate != nullptr) inv *= sigmoid_f(head_gate[(size_t)t * ldhg + head]);
    bf16_t* op = out + (size_t)t * ldo + (size_t)head * DV;
#pragma unroll
    for (int c = 0; c < CPW; ++c)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        bf16_t o4[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) o4[x] = f_to_bf16(O[c][4 * rg + x] * inv);
        *reinterpret_cast<uint2*>(op + 32 * (wave * CPW + c) + 8 * rg + 4 * h2) = *reinterpret_cast<const uint2*>(o4);
      }
  } else {
    float* pp = part + (((size_t)t * H + head) * nsplit + blockIdx.z) * (DV + 4);     // record: values[DV] | maximum | sum | pad
    if (wave == 0 && h2 == 0) { pp[DV] = m; pp[DV + 1] = l; }
#pragma unroll
    for (int c = 0; c < CPW; ++c)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg)
        *reinterpret_cast<float4*>(pp + 32 * (wave * CPW + c) + 8 * rg + 4 * h2) =
            make_float4(O[c][4 * rg], O[c][4 * rg + 1], O[c][4 * rg + 2], O[c][4 * rg + 3]);
  }
}

// -2: shape not served (the caller runs fls_seq_attn_paged)
extern "C" int fls_seq_attn_heads(const void* q, int ldq, const void* kc, int ldk, const void* vc, int ldv, void* out, int ldo,
                                  const int* tok_seq, const int* tok_pos, const int* page_table, int pt_stride, int T, int H,
                                  int G, int d, int dv, float scale, int window, int keep_first, float out_scale, int page_size,
                                  int nsplit, float* part, const float* sink_h, const float* head_gate, int ldhg, fls_stream_t s) {
  if (T <= 0) return 0;
  if (G < 1 || H % G || H / G > 32 || page_size < 1 || nsplit < 1 || nsplit > 64 || (nsplit > 1 && part == nullptr) || ldq % 4 || ldo % 4 ||
      ldk % 8 || ldv % 8 || G * d > ldk || G * dv > ldv || (uintptr_t)q % 16 || (uintptr_t)kc % 16 || (uintptr_t)vc % 16 ||
      (uintptr_t)out % 8 || keep_first < 0)
    return -2;
  const int page_shift = (page_size & (page_size - 1)) == 0 ? __builtin_ctz(page_size) : -1;
  dim3 grid(T, G, nsplit);
  hipStream_t st = (hipStream_t)s;
#define ATTN_HEADS(DD, DDV)                                                                                                \
  hipLaunchKernelGGL((attn_heads_kernel<DD, DDV>), grid, dim3(256), 0, st, (const float*)q, ldq, (const bf16_t*)kc, ldk,    \
                     (const bf16_t*)vc, ldv, (bf16_t*)out, ldo, tok_seq, tok_pos, page_table, pt_stride, H, G, scale, window, \
                     keep_first, out_scale, page_size, part, sink_h, head_gate, ldhg, page_shift)
  if (d == 576 && dv == 512) ATTN_HEADS(576, 512);
  else if (d == 512 && dv == 512) ATTN_HEADS(512, 512);
  else if (d == 256 && dv == 256) ATTN_HEADS(256, 256);
  else if (d == 128 && dv == 128) ATTN_HEADS(128, 128);
  else if (d == 320 && dv == 256) ATTN_HEADS(320, 256);
  else if (d == 192 && dv == 128) ATTN_HEADS(192, 128);
  else return -2;
#undef ATTN_HEADS
  SEQ_LAUNCH_CHECK();
  if (nsplit > 1) return seq_attn_merge(part, out, 1, ldo, T, H, dv, nsplit, 0, out_scale, sink_h != nullptr, 0.f, sink_h, head_gate, ldhg, s);
  return 0;
}
