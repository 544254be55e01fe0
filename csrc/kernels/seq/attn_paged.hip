// Attention of packed rows over paged keys and values, for prompts and for decoding alike: softmax
// over the visible keys, or (gate_bias given) every key weighted by sigmoid(score + gate_bias[h]) on its
// own.  Visible: j <= i inside the row's chunk and / or window, plus, with keep_first, the first
// keep_first keys of the sequence however far back they lie.  Keys and values are the first G d and
// G dv columns of pool rows ldk and ldv wide, so both may be one pool (values = a prefix of the keys:
// attention over latent rows).  The query may be fp32 while the pools hold bf16.  has_sink: the softmax
// has one more entry of score `sink` (sink_h given: sink_h[head]) and no value (p_j = exp(s_j) / (exp(sink) + sum exp(s))); head_gate
// [T, H] fp32: the output of (row, head) times sigmoid(head_gate[t, h]).  Pooled blocks (pool_P > 0, beside a window):
// the softmax also runs over one mean key and value for each block of pool_P positions that ends before the window,
// read from block pools with pages of their own.
//
// One block (four wavefronts) per (row, query head).  The row's query sits in LDS as fp32.  The keys
// it may see -- j <= i, inside its chunk of the sequence and / or its window -- are walked in tiles of
// 64, the four waves taking tiles in turn:
//   scores : lane = key.  The lane finds its key's row in the request's page table, reads the key
//            (16-byte loads when the head size allows) against the query in LDS, scales, caps
//            (cap * tanh(s / cap)) and subtracts the distance penalty r1 * log(1 + r2 * (i - j));
//   softmax: running maximum and sum per wave (online), weights to LDS;
//   values : heads of 32, 64, 128 or 256 aligned values (FOUR): a lane has four columns of every 64 >> vsh-th key, eight of them in
//            flight; any other: lane = value column, the lane walks the tile's keys (up to 8 x 64 columns).
// The four waves' (maximum, sum, accumulator) are merged through LDS at the end.  All of it is fp32;
// only the stored keys / values and the output have the model's element type.  A decoded token is
// one row, so its block walks the (bounded) chunk or window with four waves; a prompt has one block
// per row and head, which fills the chip without a second kernel.
//
// What bounds a decoded row is latency: a key's 16-byte loads came in two or three at a time, a value's columns 2 or 4 bytes a lane.  With
// KU of a key's 16-byte pieces and eight keys' values in flight: 16 requests of 1,000 keys, 32 heads of 128 on 8, 61.7 -> 45.6 us; 8 of 90
// .. 240, 16 heads 10.3 -> 9.4; in fp32 prompts of 400, 300 and 210 rows 217 -> 200.  What bounds many rows is how many waves a SIMD
// holds, so each form is a kernel of its own (bf16: 64 registers a lane without FOUR, 94 with KU = 4, 87 with 8; both in one 136, and
// prompts of heads of 96 took 1.4 to 1.8 times as long).  6,500 random calls, mean over the lane = column kernel by heads of values: 32
// (KU = 4) 0.64 .. 0.82, with KU = 8 0.73 .. 1.02 and up to 1.2; 64 .. 256 (KU = 8) 0.57 .. 0.86, with KU = 4 0 to 3 hundredths more; any
// other (KU = 1) the same, with KU = 8 up to 1.3.  With blocks (POOL, 4,300 calls) 32 .. 128 (KU = 4) 0.70 .. 0.89, with KU = 8 0.71 ..
// 0.89 and up to 1.2; 256 (KU = 1) 0.74 .. 0.89, with KU = 8 up to 1.3.
#include "seq_common.h"
#include "fls_seq.h"
#include "row_vec.h"

#define MAX_DV_PER_LANE 8      // value columns per lane: head value size <= 512 (a latent row)
#define MAX_D 1024

// KU pieces of 16 bytes of the row in flight, the sum in the same order
template <typename T, int KU>
__device__ __forceinline__ float dot_row(const T* __restrict__ k, const float* __restrict__ q, int d, int vec) {
  float acc = 0.f;
  if (vec) {
    if constexpr (sizeof(T) == 2) {
      int c = 0;
      for (; KU > 1 && c + 8 * KU <= d; c += 8 * KU) {
        uint4 v[KU];
#pragma unroll
        for (int x = 0; x < KU; ++x) v[x] = *reinterpret_cast<const uint4*>(k + c + 8 * x);
#pragma unroll
        for (int x = 0; x < KU; ++x) {
          const bf16_t* e = reinterpret_cast<const bf16_t*>(&v[x]);
#pragma unroll
          for (int i = 0; i < 8; ++i) acc += bf16_to_f(e[i]) * q[c + 8 * x + i];
        }
      }
      for (; c < d; c += 8) {
        const uint4 v = *reinterpret_cast<const uint4*>(k + c);
        const bf16_t* e = reinterpret_cast<const bf16_t*>(&v);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc += bf16_to_f(e[i]) * q[c + i];
      }
    } else {
      int c = 0;
      for (; KU > 1 && c + 4 * KU <= d; c += 4 * KU) {
        float4 v[KU];
#pragma unroll
        for (int x = 0; x < KU; ++x) v[x] = *reinterpret_cast<const float4*>(k + c + 4 * x);
#pragma unroll
        for (int x = 0; x < KU; ++x) acc += v[x].x * q[c + 4 * x] + v[x].y * q[c + 4 * x + 1] + v[x].z * q[c + 4 * x + 2] + v[x].w * q[c + 4 * x + 3];
      }
      for (; c < d; c += 4) {
        const float4 v = *reinterpret_cast<const float4*>(k + c);
        acc += v.x * q[c] + v.y * q[c + 1] + v.z * q[c + 2] + v.w * q[c + 3];
      }
    }
  } else {
    for (int c = 0; c < d; ++c) acc += ldf(k, c) * q[c];
  }
  return acc;
}

template <typename TQ, typename T, typename TO, bool POOL, bool FOUR, int KU>
__global__ __launch_bounds__(256) void attn_paged_kernel(const TQ* __restrict__ q, int ldq, const T* kc, int ldk,
                                                         const T* vc, int ldv, TO* __restrict__ out, int ldo,
                                                         const int* __restrict__ tok_seq, const int* __restrict__ tok_pos,
                                                         const int* __restrict__ page_table, int pt_stride, int H, int G,
                                                         int d, int dv, float scale, float softcap,
                                                         const float* __restrict__ r1, const float* __restrict__ r2,
                                                         int chunk, int window, int keep_first,
                                                         const float* __restrict__ gate_bias, float out_scale,
                                                         int page_size, int vec, int vsh, float* __restrict__ part, int has_sink,
                                                         float sink, const float* __restrict__ sink_h,
                                                         const float* __restrict__ head_gate, int ldhg, int Gv,
                                                         AttnBlocks ab) {
  __shared__ float qs[MAX_D];
  __shared__ float pw[4][64];
  __shared__ int prow[4][64];
  __shared__ float mm[4], ll[4];
  __shared__ __attribute__((aligned(16))) float accs[4][MAX_DV_PER_LANE * 64];
  const int t = blockIdx.y, h = blockIdx.x;
  const int g = h / (H / G);
  const int gv = g % Gv;                          // (several score maps over the same values: Gv < G value heads)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = tok_pos[t];
  const int* table = page_table + (size_t)tok_seq[t] * pt_stride;
  for (int c = threadIdx.x; c < d; c += 256) qs[c] = ldf(q + (size_t)t * ldq + (size_t)h * d, c);
  __syncthreads();
  int lo = chunk > 0 ? (i / chunk) * chunk : 0;
  if (window > 0 && i - window + 1 > lo) lo = i - window + 1;
  // what precedes the window's keys: kept first keys that the window no longer covers, or the seen blocks
  const int nkeep = POOL ? (i - window + 1 > 0 ? (i - window + 1) / ab.P : 0) : min(keep_first, lo);
  const int* btable = POOL ? ab.table + (size_t)tok_seq[t] * ab.t_stride : nullptr;
  const int nkeys = nkeep + i - lo + 1;
  // (with blocks every tile holds keys of one kind: nbt tiles of blocks, then tiles of tokens)
  const int nbt = POOL ? (nkeep + 63) / 64 : 0;
  const int ntiles = POOL ? nbt + (i - lo) / 64 + 1 : (nkeys + 63) / 64;
  const float a1 = r1 != nullptr ? r1[h] : 0.f, a2 = r2 != nullptr ? r2[h] : 0.f;
  const bool gated = gate_bias != nullptr;
  const float gb = gated ? gate_bias[h] : 0.f;
  const float snk = has_sink && sink_h != nullptr ? sink_h[h] : sink;
  float m = -1e30f, l = 0.f;
  constexpr int NA = FOUR ? 4 : MAX_DV_PER_LANE;
  float acc[NA];
#pragma unroll
  for (int c = 0; c < NA; ++c) acc[c] = 0.f;
  // gridDim.z > 1: the key tiles are cut into gridDim.z ranges, one block each, whose (maximum, sum,
  // weighted values) go to `part` and are merged by attn_merge_kernel
  const int nsplit = gridDim.z;
  const int tps = (ntiles + nsplit - 1) / nsplit;
  const int tile_hi = min(ntiles, ((int)blockIdx.z + 1) * tps);
  for (int tile = blockIdx.z * tps + wave; tile < tile_hi; tile += 4) {
    const bool pooled = POOL && tile < nbt;        // (wave-uniform)
    const int n = POOL ? (pooled ? tile : tile - nbt) * 64 + lane : tile * 64 + lane;
    const int tkeys = POOL ? (pooled ? nkeep : i - lo + 1) : nkeys;
    const bool valid = n < tkeys;
    const int j = POOL ? (pooled ? n : lo + n) : (n < nkeep ? n : lo + (n - nkeep));
    const int* tab = pooled ? btable : table;
    const T* kb = pooled ? reinterpret_cast<const T*>(ab.kp) : kc;
    const T* vb = (pooled ? reinterpret_cast<const T*>(ab.vp) : vc) + (size_t)gv * dv;
    const int lk = pooled ? ab.ldk : ldk, lv = pooled ? ab.ldv : ldv;
    float sc = -1e30f;
    int row = 0;
    if (valid) {
      row = tab[j / page_size] * page_size + j % page_size;
      sc = dot_row<T, KU>(kb + (size_t)row * lk + (size_t)g * d, qs, d, vec) * scale;
      if (softcap > 0.f) sc = softcap * tanhf(sc / softcap);
      if (a1 != 0.f) sc -= a1 * log1pf(a2 * (float)(i - j));
    }
    float p, corr = 1.f;
    if (gated) {
      p = valid ? sigmoid_f(sc + gb) : 0.f;
    } else {
      const float mt = fmaxf(m, wave_max(sc));
      p = valid ? expf(sc - mt) : 0.f;
      corr = expf(m - mt);
      l = l * corr + wave_sum(p);
      m = mt;
    }
    pw[wave][lane] = p;
    prow[wave][lane] = row;
    // (a wave reads back only what its own lanes wrote: LDS ordering within a wave needs no barrier,
    // but the compiler must not move the loads above the stores)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int nk = min(64, tkeys - (n - lane));
    if constexpr (FOUR) {                          // 64 >> vsh keys side by side, eight of these in flight
      const int at = 64 >> vsh, sub = lane >> vsh, col = 4 * (lane & ((1 << vsh) - 1));
#pragma unroll
      for (int x = 0; x < 4; ++x) acc[x] *= corr;
      for (int j0 = sub; j0 - sub < nk; j0 += 8 * at) {
        RowVec<4> v[8];
        float pj[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          const int jj = min(j0 + x * at, nk - 1);
          pj[x] = pw[wave][jj];
          v[x] = row_load<4>(vb + (size_t)prow[wave][jj] * lv + col);
        }
#pragma unroll
        for (int x = 0; x < 8; ++x)
          if (j0 + x * at < nk) {
#pragma unroll
            for (int y = 0; y < 4; ++y) acc[y] += pj[x] * v[x].v[y];
          }
      }
    } else {
#pragma unroll
      for (int c = 0; c < MAX_DV_PER_LANE; ++c) {
        const int e = lane + 64 * c;
        if (e < dv) {
          float a = acc[c] * corr;
          int jj = 0;
          for (; jj + 8 <= nk; jj += 8) {          // eight independent value loads in flight
            float v[8];
#pragma unroll
            for (int x = 0; x < 8; ++x) v[x] = ldf(vb + (size_t)prow[wave][jj + x] * lv, e);
#pragma unroll
            for (int x = 0; x < 8; ++x) a += pw[wave][jj + x] * v[x];
          }
          for (; jj < nk; ++jj) a += pw[wave][jj] * ldf(vb + (size_t)prow[wave][jj] * lv, e);
          acc[c] = a;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (lane == 0) { mm[wave] = m; ll[wave] = l; }
  if constexpr (FOUR) {
    for (int o = 1 << vsh; o < 64; o <<= 1)
#pragma unroll
      for (int x = 0; x < 4; ++x) acc[x] += __shfl_xor(acc[x], o, 64);
    if (lane >> vsh == 0) *reinterpret_cast<float4*>(&accs[wave][4 * lane]) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  } else {
#pragma unroll
    for (int c = 0; c < MAX_DV_PER_LANE; ++c) accs[wave][lane + 64 * c] = acc[c];
  }
  __syncthreads();
  if (wave == 0) {
    float f[4], inv = out_scale, mx = 0.f, lt = 0.f;
    if (gated) {
#pragma unroll
      for (int w = 0; w < 4; ++w) f[w] = 1.f;
    } else {
      mx = fmaxf(fmaxf(mm[0], mm[1]), fmaxf(mm[2], mm[3]));
      if (has_sink && nsplit == 1) mx = fmaxf(mx, snk);           // (with ranges the merge adds the silent entry, once)
#pragma unroll
      for (int w = 0; w < 4; ++w) { f[w] = expf(mm[w] - mx); lt += ll[w] * f[w]; }
      if (has_sink && nsplit == 1) lt += expf(snk - mx);
      inv = out_scale / lt;
    }
    if (head_gate != nullptr) inv *= sigmoid_f(head_gate[(size_t)t * ldhg + h]);
    if (nsplit > 1) {                              // this range's share, not yet normalised
      float* pp = part + (((size_t)t * H + h) * nsplit + blockIdx.z) * (dv + 4);      // record: values[dv] | maximum | sum | pad
      if (lane == 0) { pp[dv] = mx; pp[dv + 1] = lt; }
#pragma unroll
      for (int c = 0; c < MAX_DV_PER_LANE; ++c) {
        const int e = lane + 64 * c;
        if (e < dv) pp[e] = accs[0][e] * f[0] + accs[1][e] * f[1] + accs[2][e] * f[2] + accs[3][e] * f[3];
      }
      return;
    }
#pragma unroll
    for (int c = 0; c < MAX_DV_PER_LANE; ++c) {
      const int e = lane + 64 * c;
      if (e < dv) {
        const float v = accs[0][e] * f[0] + accs[1][e] * f[1] + accs[2][e] * f[2] + accs[3][e] * f[3];
        stf(out + (size_t)t * ldo + (size_t)h * dv, e, v * inv);
      }
    }
  }
}

// Few rows (decoding, some requests): what bounds a (row, head) is the chain of one tile -- its keys' page entries, the keys, the weights,
// the values, each a trip to memory -- and 64 keys a tile gave that chain 200 to 400 keys' work on four waves.  Here sixteen waves take
// tiles of 16 keys in turn: four lanes share a key, each every fourth 16-byte piece of it, all of a head of 128 in flight at once, and the
// tile's values are one or two batches of loads.  A row of fewer than 256 keys is one tile a wave.  (aligned rows, FOUR's head sizes, no
// blocks.)  us in turn, the other kernel with its ranges over twice the blocks, bf16 heads of 128: 128 rows x heads of 220 keys 9.9 ->
// 8.0, 400 15.5 -> 10.8, 1,000 21.0 -> 17.3; 48 x 400 15.3 -> 10.2, 1,000 18.2 -> 11.8; fp32 48 x 400 18.0 -> 11.7; of 210 combinations of
// 8 to 256 rows x heads, 20 to 4,000 keys, heads of 64 to 256 0.77 of the time.
template <typename TQ, typename T, typename TO>
__global__ __launch_bounds__(1024) void attn_few_kernel(const TQ* __restrict__ q, int ldq, const T* __restrict__ kc, int ldk,
                                                        const T* __restrict__ vc, int ldv, TO* __restrict__ out, int ldo,
                                                        const int* __restrict__ tok_seq, const int* __restrict__ tok_pos,
                                                        const int* __restrict__ page_table, int pt_stride, int H, int G,
                                                        int d, int dv, float scale, float softcap,
                                                        const float* __restrict__ r1, const float* __restrict__ r2,
                                                        int chunk, int window, int keep_first,
                                                        const float* __restrict__ gate_bias, float out_scale,
                                                        int page_size, int vsh, float* __restrict__ part, int has_sink,
                                                        float sink, const float* __restrict__ sink_h,
                                                        const float* __restrict__ head_gate, int ldhg, int Gv) {
  constexpr int WV = 16, KEYS = 16, PE = 16 / sizeof(T), KU = 4;      // elements of a piece, pieces in flight a lane
  __shared__ __attribute__((aligned(16))) float qs[MAX_D];
  __shared__ float pw[WV][KEYS];
  __shared__ int prow[WV][KEYS];
  __shared__ float mm[WV], ll[WV];
  __shared__ __attribute__((aligned(16))) float accs[WV][256];
  const int t = blockIdx.y, h = blockIdx.x;
  const int g = h / (H / G), gv = g % Gv;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = tok_pos[t];
  const int* table = page_table + (size_t)tok_seq[t] * pt_stride;
  for (int c = threadIdx.x; c < d; c += 64 * WV) qs[c] = ldf(q + (size_t)t * ldq + (size_t)h * d, c);
  __syncthreads();
  int lo = chunk > 0 ? (i / chunk) * chunk : 0;
  if (window > 0 && i - window + 1 > lo) lo = i - window + 1;
  const int nkeep = min(keep_first, lo), nkeys = nkeep + i - lo + 1, ntiles = (nkeys + KEYS - 1) / KEYS;
  const float a1 = r1 != nullptr ? r1[h] : 0.f, a2 = r2 != nullptr ? r2[h] : 0.f;
  const bool gated = gate_bias != nullptr;
  const float gb = gated ? gate_bias[h] : 0.f;
  const float snk = has_sink && sink_h != nullptr ? sink_h[h] : sink;
  const int key = lane >> 2, sub4 = lane & 3, pieces = d / PE;
  const int at = 64 >> vsh, sub = lane >> vsh, col = 4 * (lane & ((1 << vsh) - 1));
  float m = -1e30f, l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
  const int nsplit = gridDim.z, tps = (ntiles + nsplit - 1) / nsplit, tile_hi = min(ntiles, ((int)blockIdx.z + 1) * tps);
  for (int tile = blockIdx.z * tps + wave; tile < tile_hi; tile += WV) {
    const int n = tile * KEYS + key;
    const bool valid = n < nkeys;
    const int j = n < nkeep ? n : lo + (n - nkeep);
    float sc = 0.f;
    int row = 0;
    if (valid) {
      row = table[j / page_size] * page_size + j % page_size;
      const T* k = kc + (size_t)row * ldk + (size_t)g * d;
      for (int p0 = sub4; p0 < pieces; p0 += 4 * KU) {
        uint4 v[KU];
#pragma unroll
        for (int x = 0; x < KU; ++x) v[x] = *reinterpret_cast<const uint4*>(k + min(p0 + 4 * x, pieces - 1) * PE);
#pragma unroll
        for (int x = 0; x < KU; ++x)
          if (p0 + 4 * x < pieces) {
            const T* e = reinterpret_cast<const T*>(&v[x]);
            const float* qp = qs + (p0 + 4 * x) * PE;
#pragma unroll
            for (int y = 0; y < PE; ++y) sc += ldf(e, y) * qp[y];
          }
      }
    }
    sc += __shfl_xor(sc, 1, 64);
    sc += __shfl_xor(sc, 2, 64);
    sc *= scale;
    if (softcap > 0.f) sc = softcap * tanhf(sc / softcap);
    if (a1 != 0.f) sc -= a1 * log1pf(a2 * (float)max(i - j, 0));
    if (!valid) sc = -1e30f;
    float p, corr = 1.f;
    if (gated) {
      p = valid ? sigmoid_f(sc + gb) : 0.f;
    } else {
      const float mt = fmaxf(m, wave_max(sc));
      p = valid ? expf(sc - mt) : 0.f;
      corr = expf(m - mt);
      l = l * corr + wave_sum(sub4 == 0 ? p : 0.f);
      m = mt;
    }
    if (sub4 == 0) {
      pw[wave][key] = p;
      prow[wave][key] = row;
    }
    // (a wave reads back only what its own lanes wrote: no barrier, but the compiler must not move the loads above the stores)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int nk = min(KEYS, nkeys - tile * KEYS);
#pragma unroll
    for (int x = 0; x < 4; ++x) acc[x] *= corr;
    for (int j0 = sub; j0 - sub < nk; j0 += 8 * at) {
      RowVec<4> v[8];
      float pj[8];
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        const int jj = min(j0 + x * at, nk - 1);
        pj[x] = pw[wave][jj];
        v[x] = row_load<4>(vc + (size_t)gv * dv + (size_t)prow[wave][jj] * ldv + col);
      }
#pragma unroll
      for (int x = 0; x < 8; ++x)
        if (j0 + x * at < nk) {
#pragma unroll
          for (int y = 0; y < 4; ++y) acc[y] += pj[x] * v[x].v[y];
        }
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (lane == 0) { mm[wave] = m; ll[wave] = l; }
  for (int o = 1 << vsh; o < 64; o <<= 1)
#pragma unroll
    for (int x = 0; x < 4; ++x) acc[x] += __shfl_xor(acc[x], o, 64);
  if (lane >> vsh == 0) *reinterpret_cast<float4*>(&accs[wave][4 * lane]) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  __syncthreads();
  if (64 * wave >= dv) return;
  // (lane w & 15: wave w's maximum and sum, in each wave that writes)
  float f = 1.f, inv = out_scale, mx = 0.f, lt = 0.f;
  if (!gated) {
    const float mz = mm[lane & (WV - 1)];
    mx = wave_max(mz);
    if (has_sink && nsplit == 1) mx = fmaxf(mx, snk);
    f = expf(mz - mx);
    lt = wave_sum(lane < WV ? ll[lane & (WV - 1)] * f : 0.f);
    if (has_sink && nsplit == 1) lt += expf(snk - mx);
    inv = out_scale / lt;
  }
  if (head_gate != nullptr) inv *= sigmoid_f(head_gate[(size_t)t * ldhg + h]);
  const int e = threadIdx.x;
  float v = 0.f;
#pragma unroll
  for (int w = 0; w < WV; ++w) v += accs[w][e] * __shfl(f, w, 64);
  if (nsplit > 1) {
    float* pp = part + (((size_t)t * H + h) * nsplit + blockIdx.z) * (dv + 4);
    if (e == 0) { pp[dv] = mx; pp[dv + 1] = lt; }
    if (e < dv) pp[e] = v;
  } else if (e < dv) {
    stf(out + (size_t)t * ldo + (size_t)h * dv, e, v * inv);
  }
}

// out[t, h] from the nsplit partial results of a (row, head): softmax parts are rescaled to the common
// maximum and divided by the total sum, gated parts are added.  The nsplit weights are worked out once
// per block (nsplit <= MERGE_MAX_SPLIT), then every thread sums its value columns over the parts.
#define MERGE_MAX_SPLIT 64
template <typename T>
__global__ void attn_merge_kernel(const float* __restrict__ part, T* __restrict__ out, int ldo, int H, int dv, int nsplit, int gated,
                                  float out_scale, int has_sink, float sink, const float* __restrict__ sink_h,
                                  const float* __restrict__ head_gate, int ldhg) {
  __shared__ float wz[MERGE_MAX_SPLIT];
  const int t = blockIdx.y, h = blockIdx.x;
  const int rs = dv + 4;                           // record: values[dv] | maximum | sum | pad
  const float* pp = part + ((size_t)t * H + h) * nsplit * rs;
  if (threadIdx.x < 64) {                          // (one wave: lane z holds part z's maximum and sum)
    const int z = threadIdx.x;
    const float mz = (z < nsplit && !gated) ? pp[z * rs + dv] : -1e30f;
    const float lz = (z < nsplit && !gated) ? pp[z * rs + dv + 1] : 0.f;
    float mx = wave_max(mz);
    const float snk = has_sink && sink_h != nullptr ? sink_h[h] : sink;
    if (has_sink) mx = fmaxf(mx, snk);
    const float f = expf(mz - mx);
    float lt = wave_sum(lz * f);
    if (has_sink) lt += expf(snk - mx);
    const float os = head_gate != nullptr ? out_scale * sigmoid_f(head_gate[(size_t)t * ldhg + h]) : out_scale;
    wz[z] = gated ? os : f * os / lt;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < dv; e += blockDim.x) {
    float v = 0.f;
    for (int z = 0; z < nsplit; ++z) v += pp[z * rs + e] * wz[z];
    stf(out + (size_t)t * ldo + (size_t)h * dv, e, v);
  }
}

// (also used by the matrix-core kernels that cut a row's keys over blocks)
int seq_attn_merge(const float* part, void* out, int tc, int ldo, int T, int H, int dv, int nsplit, int gated, float out_scale,
                   int has_sink, float sink, const float* sink_h, const float* head_gate, int ldhg, fls_stream_t s) {
  const int threads = dv > 128 ? 256 : (dv > 64 ? 128 : 64);
  hipStream_t st = (hipStream_t)s;
  if (tc == 1) hipLaunchKernelGGL((attn_merge_kernel<bf16_t>), dim3(H, T), dim3(threads), 0, st, part, (bf16_t*)out, ldo, H, dv, nsplit, gated, out_scale, has_sink, sink, sink_h, head_gate, ldhg);
  else hipLaunchKernelGGL((attn_merge_kernel<float>), dim3(H, T), dim3(threads), 0, st, part, (float*)out, ldo, H, dv, nsplit, gated, out_scale, has_sink, sink, sink_h, head_gate, ldhg);
  SEQ_LAUNCH_CHECK();
  return 0;
}

// lanes (a power of two, as an exponent) that share a row of values, four columns each; -1: not so many columns or not so aligned
static int value_lanes(const void* vc, int ldv, int es, int dv) {
  if ((uintptr_t)vc % (4 * es) || ldv % 4) return -1;
  return dv == 32 ? 3 : dv == 64 ? 4 : dv == 128 ? 5 : dv == 256 ? 6 : -1;
}
static bool keys_by_16(const void* kc, int ldk, int es, int d) { return d * es % 16 == 0 && (uintptr_t)kc % 16 == 0 && ldk * es % 16 == 0; }
// Sixteen waves a (row, head) and range of its keys?  One block a CU (a second one waits: 384 and 512 blocks 1.0 to 1.4 of the other
// kernel's time) and keys of 256 bytes or more (128 bytes are two loads a lane here and eight there: 0.9 to 1.2)
static bool few_rows(const void* kc, int ldk, const void* vc, int ldv, int es, int d, int dv, int pool_P, long long blocks) {
  return pool_P == 0 && blocks <= 256 && d * es >= 256 && keys_by_16(kc, ldk, es, d) && value_lanes(vc, ldv, es, dv) >= 0;
}

// Ranges of keys for rows of up to `bound` keys: of 256 keys or more, so many that the launch has a block a CU of sixteen waves, or two of four
extern "C" int fls_seq_attn_ranges(const void* kc, int ldk, const void* vc, int ldv, int tc, int T, int H, int d, int dv, int pool_P, int bound) {
  const long long rows = (long long)T * H;
  if (rows < 1) return 1;
  const long long n = (few_rows(kc, ldk, vc, ldv, tc == 1 ? 2 : 4, d, dv, pool_P, rows) ? 256 : 512) / rows;
  return max(1, min(min(8, (int)n), pool_P == 0 ? bound / 256 : (bound + 255) / 256));
}

// tq: type of q; tc: type of the pools; to: type of out (fp32 over bf16 pools allowed)
extern "C" int fls_seq_attn_paged(const void* q, int ldq, int tq, const void* kc, int ldk, const void* vc, int ldv, int tc,
                                  void* out, int to, int ldo, const int* tok_seq, const int* tok_pos, const int* page_table,
                                  int pt_stride, int T, int H, int G, int d, int dv, float scale, float softcap,
                                  const float* r1, const float* r2, int chunk, int window, int keep_first,
                                  const float* gate_bias, float out_scale, int page_size, int nsplit, float* part,
                                  int has_sink, float sink, const float* sink_h, const float* head_gate, int ldhg, int Gv, int pool_P, const void* kp,
                                  int ldkp, const void* vp, int ldvp, const int* block_table, int bt_stride, fls_stream_t s) {
  if (T <= 0) return 0;
  if (Gv <= 0) Gv = G;
  if (G % Gv || (to == 1 && tc == 0)) return -1;
  if (has_sink && gate_bias != nullptr) return -1;      // (a silent entry belongs to a softmax)
  if (nsplit < 1 || nsplit > MERGE_MAX_SPLIT || (nsplit > 1 && part == nullptr)) return -1;
  if (d > MAX_D || dv > 64 * MAX_DV_PER_LANE || G < 1 || H % G || page_size < 1 || G * d > ldk || Gv * dv > ldv || keep_first < 0
      || (tq == 1 && tc == 0)) return -1;
  if (pool_P < 0 || (pool_P > 0 && (window < 1 || chunk > 0 || keep_first > 0 || has_sink || gate_bias != nullptr || r1 != nullptr ||
                                    kp == nullptr || vp == nullptr || block_table == nullptr || G * d > ldkp || Gv * dv > ldvp)))
    return -1;                                          // (blocks go with a plain softmax over a window)
  const AttnBlocks ab = {pool_P, kp, ldkp, vp, ldvp, block_table, bt_stride};
  dim3 grid(H, T, nsplit);
  hipStream_t st = (hipStream_t)s;
  const int es = tc == 1 ? 2 : 4;
  const int vsh = pool_P == 0 || value_lanes(vp, ldvp, es, dv) >= 0 ? value_lanes(vc, ldv, es, dv) : -1;
  const int vec = keys_by_16(kc, ldk, es, d) && (pool_P == 0 || keys_by_16(kp, ldkp, es, d));
  const bool few = few_rows(kc, ldk, vc, ldv, es, d, dv, pool_P, (long long)T * H * nsplit);
#define ATTN_PAGED_ARGS ldq, (const TC*)kc, ldk, (const TC*)vc, ldv, (TOUT*)out, ldo, tok_seq, tok_pos, page_table, pt_stride, H, G, \
                        d, dv, scale, softcap, r1, r2, chunk, window, keep_first, gate_bias, out_scale, page_size, vec, vsh, part, has_sink, sink, sink_h, \
                        nsplit > 1 ? nullptr : head_gate, ldhg, Gv, ab
#define ATTN_PAGED_FORM(TQ, POOL, FOUR, KU) \
  hipLaunchKernelGGL((attn_paged_kernel<TQ, TC, TOUT, POOL, FOUR, KU>), grid, dim3(256), 0, st, (const TQ*)q, ATTN_PAGED_ARGS)
#define ATTN_PAGED_GO(TQ)                                         \
  do {                                                            \
    if (few) {                                                    \
      hipLaunchKernelGGL((attn_few_kernel<TQ, TC, TOUT>), grid, dim3(1024), 0, st, (const TQ*)q, ldq, (const TC*)kc, ldk, (const TC*)vc, ldv, (TOUT*)out, ldo, \
                         tok_seq, tok_pos, page_table, pt_stride, H, G, d, dv, scale, softcap, r1, r2, chunk, window, keep_first, gate_bias, out_scale, page_size, \
                         vsh, part, has_sink, sink, sink_h, nsplit > 1 ? nullptr : head_gate, ldhg, Gv); \
    } else if (pool_P > 0) {                                      \
      if (vsh < 0) ATTN_PAGED_FORM(TQ, true, false, 1);           \
      else if (dv == 256) ATTN_PAGED_FORM(TQ, true, true, 1);     \
      else ATTN_PAGED_FORM(TQ, true, true, 4);                    \
    } else if (vsh < 0) ATTN_PAGED_FORM(TQ, false, false, 1);     \
    else if (dv == 32) ATTN_PAGED_FORM(TQ, false, true, 4);       \
    else ATTN_PAGED_FORM(TQ, false, true, 8);                     \
  } while (0)
  if (tc == 1) {
    using TC = bf16_t;
    if (to == 0) {
      using TOUT = float;
      if (tq == 1) ATTN_PAGED_GO(bf16_t);
      else ATTN_PAGED_GO(float);
    } else {
      using TOUT = bf16_t;
      if (tq == 1) ATTN_PAGED_GO(bf16_t);
      else ATTN_PAGED_GO(float);
    }
  } else {
    using TC = float;
    using TOUT = float;
    ATTN_PAGED_GO(float);
  }
#undef ATTN_PAGED_GO
#undef ATTN_PAGED_FORM
#undef ATTN_PAGED_ARGS
  SEQ_LAUNCH_CHECK();
  if (nsplit > 1) return seq_attn_merge(part, out, to, ldo, T, H, dv, nsplit, gate_bias != nullptr, out_scale, has_sink, sink, sink_h, head_gate, ldhg, s);
  return 0;
}
