// RoPE table, query absorption and the stage-2 merge: the small kernels around the scans.
#include <algorithm>
#include <type_traits>

#include "xkv_common.h"
#include "merge_rule.h"

namespace xkv {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// ----------------------------------------------------------------------------------------------
// RoPE table.  angle = float(pos) * inv_freq[j] in fp32 (one rounding), then sincosf with full
// range reduction - the eager closed form of the reference (rope/rope_ref.py:3-9), not the
// fast-math pow/sin/cos of its Triton table kernel.
// ----------------------------------------------------------------------------------------------
template <typename O>
__global__ void rope_table_kernel(O* __restrict__ sin_out, O* __restrict__ cos_out,
                                  const float* __restrict__ inv_freq, int64_t seqlen, int64_t start,
                                  int half_dim) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= seqlen * half_dim) return;
  int j = (int)(idx % half_dim);
  int64_t l = idx / half_dim;
  float ang = (float)(start + l) * inv_freq[j];
  float s, c;
  sincosf(ang, &s, &c);
  sin_out[idx] = (O)s;
  cos_out[idx] = (O)c;
}

// ----------------------------------------------------------------------------------------------
// Rotate-half RoPE applied to rows x[b, r, h, :] at position (positions ? positions[b] : pos0) + r: one thread per pair
// (j, j + dim/2), fp32 angle float(pos) * inv_freq[j] and fp32 arithmetic as in the eager form (rope/rope_ref.py:3-20).
// ----------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void rope_apply_kernel(const T* __restrict__ x, T* __restrict__ out,
                                                          const float* __restrict__ inv_freq,
                                                          const int64_t* __restrict__ positions, int64_t pos0, int64_t total,
                                                          int rows, int heads, int half, int64_t sxb, int64_t sxr, int64_t sxh,
                                                          int64_t sob, int64_t sor, int64_t soh) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int j = (int)(idx % half);
  int64_t t = idx / half;
  const int h = (int)(t % heads);
  t /= heads;
  const int r = (int)(t % rows);
  const int64_t b = t / rows;
  const int64_t pos = (positions ? positions[b] : pos0) + r;
  float s, c;
  sincosf((float)pos * inv_freq[j], &s, &c);
  const T* xi = x + b * sxb + r * sxr + h * sxh;
  T* oi = out + b * sob + r * sor + h * soh;
  const float x0 = (float)xi[j], x1 = (float)xi[j + half];
  oi[j] = (T)(x0 * c - x1 * s);
  oi[j + half] = (T)(x1 * c + x0 * s);
}

// ----------------------------------------------------------------------------------------------
// qt[b,h,rho] = sum_d q[b,h,d] * B[b,h/G,rho,d]; one workgroup per (kv head, batch), one thread
// per rho (strided), the G query rows of the kv head held in LDS as fp32.
// ----------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void absorb_q_kernel(
    const T* __restrict__ q, const T* __restrict__ B, T* __restrict__ qt_hi, T* __restrict__ qt_lo,
    int hq, int hkv, int d, int rank, int64_t sBb, int64_t sBh, int64_t sBr) {
  typedef typename Elem<T>::vec8 vec8;
  __shared__ float qs[32 * 256];
  const int kh = blockIdx.x, b = blockIdx.y, Gall = hq / hkv;
  const int HC = 8192 / d < 32 ? 8192 / d : 32;   // heads whose query rows fit the LDS buffer at a time
  const T* Bh = B + b * sBb + kh * sBh;
  for (int gc = 0; gc < Gall; gc += HC) {
  const int G = Gall - gc < HC ? Gall - gc : HC;
  const T* qb = q + ((int64_t)b * hq + (int64_t)kh * Gall + gc) * d;
  __syncthreads();
  for (int i = threadIdx.x; i < G * d; i += blockDim.x) qs[i] = to_f32(qb[i]);
  __syncthreads();
  for (int rho = blockIdx.z * blockDim.x + threadIdx.x; rho < rank; rho += blockDim.x * gridDim.z) {
    const T* row = Bh + rho * sBr;
    for (int g0 = 0; g0 < G; g0 += 4) {
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
      for (int c = 0; c < d; c += 8) {
        vec8 v = ld16<vec8>(row + c);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float x = to_f32(v[e]);
#pragma unroll
          for (int gi = 0; gi < 4; ++gi)
            if (g0 + gi < G) acc[gi] += x * qs[(g0 + gi) * d + c + e];
        }
      }
#pragma unroll
      for (int gi = 0; gi < 4; ++gi)
        if (g0 + gi < G) {
          int64_t o = ((int64_t)b * hq + (int64_t)kh * Gall + gc + g0 + gi) * rank + rho;
          T hi = from_f32<T>(acc[gi]);
          qt_hi[o] = hi;
          if (qt_lo) qt_lo[o] = from_f32<T>(acc[gi] - to_f32(hi));
        }
    }
  }
  }
}

// The same product for every head_dim that is a multiple of 32, on v_mfma_f32_16x16x32: both operands are rows whose 8
// consecutive features are a lane's packet (A = 16 query heads, B = 16 rows of B), so they go from global memory straight into
// the matrix pipe.  A wave owns 16 rows of B against all (up to 16 per workgroup) query heads of its kv head; with KSPLIT the
// four waves of a workgroup share 16 rows and cut the features between them, so that a wave's loads are one round trip at
// d 512 too.  The kernel is latency - a launch and a round trip - whatever the shape: by trace 3.5 us at 8 x 32 heads, d 128,
// rank 512 (the LDS form it replaces: 4.4) and 4.6 us at 8 x 16 heads, d 512, rank 256 (15.5; 6.3 without KSPLIT).
template <typename T, bool KSPLIT>
__device__ __forceinline__ void absorb_q_mfma(
    const T* __restrict__ q, const T* __restrict__ B, T* __restrict__ qt_hi, T* __restrict__ qt_lo,
    int hq, int hkv, int d, int rank, int64_t sBb, int64_t sBh, int64_t sBr, int head_block, int b, int rank_block) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int NK = KSPLIT ? 4 : 8;   // k-steps in flight
  __shared__ f32x4 part[KSPLIT ? 3 : 1][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n16 = lane & 15, g4 = lane >> 4;
  const int G = hq / hkv, nhb = (G + 15) / 16;
  const int kh = head_block / nhb, g0 = (head_block % nhb) * 16;
  const int rho = (KSPLIT ? rank_block : rank_block * 4 + wave) * 16 + n16;
  const int gn = G - g0 < 16 ? G - g0 : 16;
  // head rows past the group and rows past the rank repeat the last one: their products are never written
  const T* qrow = q + ((int64_t)b * hq + (int64_t)kh * G + g0 + (n16 < gn ? n16 : gn - 1)) * d + 8 * g4;
  const T* brow = B + b * sBb + kh * sBh + (int64_t)(rho < rank ? rho : rank - 1) * sBr + 8 * g4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = KSPLIT ? 32 * NK * wave : 0; c0 < d; c0 += 32 * NK * (KSPLIT ? 4 : 1)) {
    vec8 a[NK], w[NK];
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      a[k] = w[k] = vec8{0, 0, 0, 0, 0, 0, 0, 0};
      if (c0 + 32 * k < d) {
        a[k] = ld16<vec8>(qrow + c0 + 32 * k);
        w[k] = ld16<vec8>(brow + c0 + 32 * k);
      }
    }
#pragma unroll
    for (int k = 0; k < NK; ++k) acc = Elem<T>::mfma16(a[k], w[k], acc);
  }
  if constexpr (KSPLIT) {
    if (wave) part[wave - 1][lane] = acc;
    __syncthreads();
    if (wave) return;
    acc += part[0][lane] + part[1][lane] + part[2][lane];
  }
  if (rho >= rank) return;
  // lane (n16 = row of B, g4): heads g0 + 4 g4 + r
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * g4 + r < gn) {
      const int64_t o = ((int64_t)b * hq + (int64_t)kh * G + g0 + 4 * g4 + r) * rank + rho;
      const T hi = from_f32<T>(acc[r]);
      qt_hi[o] = hi;
      if (qt_lo) qt_lo[o] = from_f32<T>(acc[r] - to_f32(hi));
    }
}

template <typename T, bool KSPLIT>
__global__ __launch_bounds__(256) void absorb_q_mfma_kernel(
    const T* __restrict__ q, const T* __restrict__ B, T* __restrict__ qt_hi, T* __restrict__ qt_lo,
    int hq, int hkv, int d, int rank, int64_t sBb, int64_t sBh, int64_t sBr) {
  absorb_q_mfma<T, KSPLIT>(q, B, qt_hi, qt_lo, hq, hkv, d, rank, sBb, sBh, sBr, blockIdx.x, blockIdx.y, blockIdx.z);
}

// ----------------------------------------------------------------------------------------------
// Prefix + tail decode starts with two things that do not depend on each other and leave most of the device idle: the query's absorption
// for the prefix, and the attention over the plain tail of recently decoded tokens.  One launch does both: the first
// `absorbing` workgroups absorb, the others take a split of the tail each, all heads of a group of at most 32.
// A tail workgroup: `tiles` tiles of 32 tokens with a running maximum.  Scores on v_mfma_f32_16x16x32, a wave for 16 tokens x 16 heads, operands
// straight from memory; the value tile goes through the LDS and is read transposed.  A launch saved is 5 - 9 us of prefix + tail calls that
// take 29 (3033 + 97 tokens, 8 heads; 22 with both launches saved) to 115 us (262144 + 128; 111); the splits of the tail, four before, are as many as the tail has tiles, up to
// 32: 4 x (20780 + 1822) tokens spent 35 us in four workgroups per sequence (88 us a call, now 68).
// ----------------------------------------------------------------------------------------------
struct TailParams {
  const void* k; const void* v;
  int64_t sKb, sKl, sVb, sVl;
  float* partial; float* lse;        // [batch, hq, splits, dv], [batch, hq, splits]
  int len, splits, tiles, groups, dv, absorbing, head_blocks, rank_blocks;
  float sm_scale, logit_cap;
};
__device__ __forceinline__ s16x4 tail_tr4(const unsigned char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
}
template <typename T, bool KSPLIT>
__global__ __launch_bounds__(256) void absorb_tail_kernel(
    const T* __restrict__ q, const T* __restrict__ B, T* __restrict__ qt_hi, T* __restrict__ qt_lo,
    int hq, int hkv, int d, int rank, int64_t sBb, int64_t sBh, int64_t sBr, const TailParams t) {
  typedef typename Elem<T>::vec8 vec8;
  if ((int)blockIdx.x < t.absorbing) {
    const int i = blockIdx.x, hb = i % t.head_blocks, b = i / t.head_blocks / t.rank_blocks;
    absorb_q_mfma<T, KSPLIT>(q, B, qt_hi, qt_lo, hq, hkv, d, rank, sBb, sBh, sBr, hb, b, i / t.head_blocks % t.rank_blocks);
    return;
  }
  constexpr int SP = 32 + 4, LDP = 32 + 8, NVB = 8, NK = KSPLIT ? 16 : 8;
  __shared__ float s_lds[32][SP];
  __shared__ T p_lds[32][LDP];
  __shared__ float a_lds[32], l_lds[32];
  extern __shared__ __attribute__((aligned(16))) unsigned char vtile[];   // [32 tokens][dv + 8]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n16 = lane & 15, g4 = lane >> 4;
  const int j = blockIdx.x - t.absorbing, split = j % t.splits, group = j / t.splits % t.groups, b = j / t.splits / t.groups;
  const int hg = hq / t.groups, h0 = group * hg;
  const int start = split * t.tiles * 32, end = min(t.len, start + t.tiles * 32), last = end - 1;
  const int tb = wave & 1, hb = wave >> 1, head = hb * 16 + n16;
  // head rows past the group and tokens past the end repeat the last ones: never written, or weighted by zero
  const T* qrow = q + ((int64_t)b * hq + h0 + (head < hg ? head : hg - 1)) * d + 8 * g4;
  vec8 w[NK];                                        // k-steps past the width multiply zeros
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    w[k] = ld16<vec8>(qrow + min(32 * k, d - 32));
    if (32 * k >= d) w[k] = vec8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  const T* kb = reinterpret_cast<const T*>(t.k) + b * t.sKb + 8 * g4;
  const T* vb = reinterpret_cast<const T*>(t.v) + b * t.sVb;
  const int vrow_bytes = t.dv * 2 + 16, nvb = t.dv / 64;
  const int srow = tid >> 3, ssub = tid & 7;
  float m_run = NEG_INF, l_run = 0.f;
  f32x4 acc[NVB][2];
#pragma unroll
  for (int mb = 0; mb < NVB; ++mb) acc[mb][0] = acc[mb][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int base = start; base < end; base += 32) {
    if (base > start) __syncthreads();               // the tile before has been read
    // every load of the tile under way before the first is waited for: a tile is one round trip
    vec8 vreg[8], a[NK];
#pragma unroll
    for (int i = 0; i < 8; ++i)                      // eight threads a row
      vreg[i] = ld16<vec8>(vb + (int64_t)min(base + srow, last) * t.sVl + (ssub + 8 * min(i, nvb - 1)) * 8);
    const int tok = base + tb * 16 + n16;
    const T* krow = kb + (int64_t)(tok < last ? tok : last) * t.sKl;
#pragma unroll
    for (int k = 0; k < NK; ++k) a[k] = ld16<vec8>(krow + min(32 * k, d - 32));
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NK; ++k) s = Elem<T>::mfma16(a[k], w[k], s);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < nvb) st16(vtile + srow * vrow_bytes + (ssub + 8 * i) * 16, vreg[i]);
    if (hb * 16 < hg) *reinterpret_cast<f32x4*>(&s_lds[head][tb * 16 + 4 * g4]) = s;   // lane (head n16, g4): tokens 4 g4 + r
    __syncthreads();
    if (srow < hg) {                                  // 8 threads a head, 4 tokens each
      float sv[4], mx = NEG_INF, sum = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = s_lds[srow][ssub * 4 + i] * t.sm_scale;
        if (t.logit_cap > 0.f) x = t.logit_cap * tanhf(x / t.logit_cap);
        sv[i] = base + ssub * 4 + i < end ? x : NEG_INF;
        mx = fmaxf(mx, sv[i]);
      }
      const float m_new = fmaxf(m_run, row_reduce<true, 8>(mx)), alpha = __expf(m_run - m_new);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __expf(sv[i] - m_new);
        sum += e;
        p_lds[srow][ssub * 4 + i] = from_f32<T>(e);
      }
      l_run = l_run * alpha + row_reduce<false, 8>(sum);
      m_run = m_new;
      if (ssub == 0) a_lds[srow] = alpha;
    }
    __syncthreads();
    // every wave a quarter of the features
#pragma unroll
    for (int hb2 = 0; hb2 < 2; ++hb2)
      if (hb2 * 16 < hg) {
        const int row = hb2 * 16 + n16 < hg ? hb2 * 16 + n16 : hg - 1;
        const float al = a_lds[row];
        const vec8 pb = ld16<vec8>(&p_lds[row][8 * g4]);
        const unsigned char* vrow = vtile + (8 * g4 + (n16 >> 2)) * vrow_bytes + (wave * (t.dv / 4) + 4 * (n16 & 3)) * 2;
#pragma unroll
        for (int mb = 0; mb < NVB; ++mb)
          if (mb < nvb) {
            const s16x8 a = __builtin_shufflevector(tail_tr4(vrow + mb * 32), tail_tr4(vrow + mb * 32 + 4 * vrow_bytes), 0, 1, 2, 3, 4, 5, 6, 7);
            acc[mb][hb2] = Elem<T>::mfma16(__builtin_bit_cast(vec8, a), pb, acc[mb][hb2] * al);
          }
      }
  }
  if (srow < hg && ssub == 0) {
    l_lds[srow] = l_run;
    t.lse[((int64_t)b * hq + h0 + srow) * t.splits + split] = m_run + __logf(l_run);
  }
  __syncthreads();
#pragma unroll
  for (int hb2 = 0; hb2 < 2; ++hb2) {
    const int h = hb2 * 16 + n16;
    if (h < hg) {
      const float inv = 1.f / l_lds[h];
      float* dst = t.partial + (((int64_t)b * hq + h0 + h) * t.splits + split) * t.dv + wave * (t.dv / 4) + 4 * g4;
#pragma unroll
      for (int mb = 0; mb < NVB; ++mb)
        if (mb < nvb) *reinterpret_cast<f32x4*>(dst + mb * 16) = acc[mb][hb2] * inv;
    }
  }
}

// ----------------------------------------------------------------------------------------------
// Block-diagonal query: out[b, h, kh * d + c] = q[b, h, c] if kh == h / G else 0.  With it the per-head keys of a token,
// stored side by side ([batch, kv_len, hkv * d]), act as ONE wide row shared by every head, so a single workgroup can
// serve all query heads of a sequence (and read a value basis shared by the heads once instead of once per kv head).
// ----------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void blockdiag_q_kernel(const T* __restrict__ q, T* __restrict__ out, int hq, int hkv, int d,
                                                          int64_t total8) {
  typedef typename Elem<T>::vec8 vec8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;   // one 8-element packet of out
  if (i >= total8) return;
  const int ppr = hkv * d / 8, dp = d / 8;
  const int64_t row = i / ppr;            // b * hq + h
  const int pk = (int)(i - row * ppr);
  const int kh = pk / dp, c = (pk - kh * dp) * 8;
  const int h = (int)(row % hq), G = hq / hkv;
  vec8 v = {0, 0, 0, 0, 0, 0, 0, 0};
  if (kh == h / G) v = ld16<vec8>(q + row * d + c);
  st16(out + i * 8, v);
}

// ----------------------------------------------------------------------------------------------
// Stage 2: weights w_i = exp(lse_i - max lse) / sum over the live splits (a prefix of the split range: split i is live iff
// per * i < L), weighted sum of the partial rows, optionally the up-projection by vB[b, kh].  Both kernels are chains of
// dependent round trips, so each starts everything it can at once: the lse words and the partial rows of a thread's splits
// are loaded together and folded with a running maximum, instead of weights first and rows after.
// ----------------------------------------------------------------------------------------------
// A thread's share of one head's splits: i = first, first + step, ... < nlive, P consecutive features at pp.  Eight splits'
// loads in flight; acc = sum exp(lse_i - m) * partial_i, l = sum exp(lse_i - m), m the running maximum (NEG_INF: no split).
template <int P> struct MergeAcc { float m, l, acc[P]; };
template <int P>
__device__ __forceinline__ MergeAcc<P> merge_fold(const float* __restrict__ pl, const float* __restrict__ pp, int dv, int first,
                                                  int step, int nlive) {
  MergeAcc<P> r;
  r.m = NEG_INF; r.l = 0.f;
#pragma unroll
  for (int e = 0; e < P; ++e) r.acc[e] = 0.f;
  constexpr int NB = 8;
  for (int i0 = first; i0 < nlive; i0 += NB * step) {
    float w[NB], v[NB][P];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int i = i0 + k * step;
      w[k] = NEG_INF;
#pragma unroll
      for (int e = 0; e < P; ++e) v[k][e] = 0.f;
      if (i < nlive) {
        w[k] = pl ? pl[i] : 0.f;
        const float* src = pp + (int64_t)i * dv;
        if constexpr (P == 4) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(src);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[k][e] = x[e];
        } else {
          v[k][0] = src[0];
        }
      }
    }
    float mn = r.m;
#pragma unroll
    for (int k = 0; k < NB; ++k) mn = fmaxf(mn, w[k]);
    const float sc = r.m == NEG_INF ? 0.f : __expf(r.m - mn);
    r.m = mn;
    r.l *= sc;
#pragma unroll
    for (int e = 0; e < P; ++e) r.acc[e] *= sc;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const float x = w[k] == NEG_INF ? 0.f : __expf(w[k] - mn);
      r.l += x;
#pragma unroll
      for (int e = 0; e < P; ++e) r.acc[e] += x * v[k][e];
    }
  }
  return r;
}

// Without an up-projection: one workgroup per (head, block of `chunk` features), chunk / P lanes per group of threads; the
// groups take the splits round-robin and meet in the LDS.  Short chunks when there are many splits, so that a single long
// sequence is read by the whole chip: batch 1, 32 heads, 256 splits of 512 features (16.8 MB) in 6.0 us by trace, 64 x 16 heads
// with 4 splits of 512 in 4.5 (with the weights of all splits first and the rows after them: 8.6).
template <typename O, int P>
__global__ __launch_bounds__(256) void merge_rows_kernel(
    const float* __restrict__ partial, const float* __restrict__ lse, O* __restrict__ out,
    const int32_t* __restrict__ num_kv_splits, const int32_t* __restrict__ kv_lens, int hq, int kv_len, int max_splits, int dv,
    int chunk, int64_t sOb, int64_t sOh, float* __restrict__ lse_out, int64_t sLb, int64_t sLh, int split_cap,
    const int32_t* __restrict__ split_plan) {
  __shared__ float red[256 * P], ml[256][2];
  const int h = blockIdx.x, b = blockIdx.y, c0 = blockIdx.z * chunk;
  const int L = kv_lens ? kv_lens[b] : kv_len;
  const int nlive = live_splits(L, effective_splits(L, asked_splits(num_kv_splits, b, max_splits, split_cap), split_cap_in_force(split_cap, split_plan)), max_splits);
  const int lanes = chunk / P, ngrp = 256 / lanes;          // lanes <= 256
  const int sg = threadIdx.x / lanes, c = c0 + (threadIdx.x % lanes) * P;
  const bool mine = sg < ngrp && c < dv;
  const PartialRows rows = partial_rows(b, hq, max_splits, num_kv_splits, split_plan);
  const int64_t row = rows.base + (int64_t)h * rows.per_head;
  MergeAcc<P> a;
  if (mine) {
    a = merge_fold<P>(lse + row, partial + row * dv + c, dv, sg, ngrp, nlive);
#pragma unroll
    for (int e = 0; e < P; ++e) red[threadIdx.x * P + e] = a.acc[e];
    ml[threadIdx.x][0] = a.m;
    ml[threadIdx.x][1] = a.l;
  }
  __syncthreads();
  if (!mine || sg) return;
  float M = a.m;
  for (int g = 1; g < ngrp; ++g) M = fmaxf(M, ml[g * lanes + threadIdx.x][0]);
  float l = 0.f, acc[P];
#pragma unroll
  for (int e = 0; e < P; ++e) acc[e] = 0.f;
  for (int g = 0; g < ngrp; ++g) {
    const int t = g * lanes + threadIdx.x;
    const float w = ml[t][0] == NEG_INF ? 0.f : __expf(ml[t][0] - M);
    l += w * ml[t][1];
#pragma unroll
    for (int e = 0; e < P; ++e) acc[e] += w * red[t * P + e];
  }
  const float inv = nlive > 0 ? 1.f / l : 0.f;
  O* o = out + b * sOb + h * sOh + c;
#pragma unroll
  for (int e = 0; e < P; ++e) o[e] = (O)(acc[e] * inv);
  if (lse_out && c == 0) lse_out[b * sLb + h * sLh] = M + __logf(l);   // log-sum-exp of the merged range
}

// With an up-projection: one workgroup per (hpw heads of one kv head, block of 64 output columns).  Thread (cb, grp): 8 columns
// x the vB rows grp, grp + 64, ...; its vB packets are on the way before the split counts are known.  The heads' merged rows
// meet in the LDS (every column block repeats that merge: a caller with many splits merges the rows first), then 8 FMAs per packet and head, and the 64 row groups are added by halving exchanges inside a 16-lane row (each step
// a lane keeps half of its sums and hands the other half over) and four LDS words per total.  Batch 1, one row per
// head, dv 512: 4.8 us in a graph of merges for 32 heads on 8 or 1 kv heads (5.8 with four heads a workgroup); 16 x 32 heads, 2 splits of 512, 8.6 us by trace (11.6).
//
// MANY_LOOP: many splits on a chip that the heads fill (launch_merge): a workgroup folds once for several column blocks.  MANY_SPREAD: on
// one that is not full: one head per workgroup, its splits dealt out among groups of threads as in merge_rows_kernel, the product for that head alone (with three
// absent heads multiplied beside it 0.6 - 0.9 us more).  ONE_HEAD: the same product where there are few splits (merge_rule.h).  32 splits of 256, 32 heads, d_out 128: 4.9 us (6.3 with a thread folding all splits of its packet), 128 of 512 9.5 (18.1).
constexpr int MERGE_UP_T = 512;
enum { ONE_PASS = 0, MANY_LOOP = 1, MANY_SPREAD = 2, ONE_HEAD = 3 };
//
// TAIL: the up-projected row is merged with rows that are in output space already (the plain tail beside a factorised prefix), by their
// log-sum-exps.  Their packets are folded while the merged rows are; a kernel of its own for it was 4 - 5 us more.
struct MergeTail { const float* partial; const float* lse; int splits; };   // [batch, hq, splits, d_out], [batch, hq, splits]
template <typename O, typename TB, int RPT, int MANY, bool TAIL>
__global__ __launch_bounds__(MERGE_UP_T) void merge_up_kernel(
    const float* __restrict__ partial, const float* __restrict__ lse, O* __restrict__ out,
    const TB* __restrict__ vB, int64_t sVb, int64_t sVh, int64_t sVr, int d_out,
    const int32_t* __restrict__ num_kv_splits, const int32_t* __restrict__ kv_lens,
    int hq, int hkv, int kv_len, int max_splits, int dv, int64_t sOb, int64_t sOh, int hpw,
    float* __restrict__ lse_out, int64_t sLb, int64_t sLh, int split_cap, const int32_t* __restrict__ split_plan, const MergeTail tail) {
  typedef typename Elem<TB>::vec8 vec8;
  extern __shared__ float merged[];               // [hpw][dv]; MANY_SPREAD: then a packet, a maximum and a sum of every thread
  constexpr int HP = MANY == MANY_SPREAD || MANY == ONE_HEAD ? 1 : 4;   // heads of a pass
  __shared__ float tot[4][HP * MERGE_CB];         // [quarter of the row groups][heads x 64 columns]
  const int hfirst = blockIdx.x * hpw, kh = hfirst / (hq / hkv), b = blockIdx.y;
  int c0 = blockIdx.z * MERGE_CB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // the 16 lanes of a row hold 16 row groups of one 8-column block; a wave covers four blocks, a pair of waves all eight
  const int cb = (wave & 1) * 4 + (lane >> 4), grp = (wave >> 1) * 16 + (lane & 15);
  const TB* Bh = vB + b * sVb + kh * sVh + cb * 8;
  vec8 w[RPT];
  auto load_w = [&]() {
    const bool cols = c0 + cb * 8 < d_out;        // d_out is a multiple of 8
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      w[r] = vec8{0, 0, 0, 0, 0, 0, 0, 0};
      if (cols && grp + 64 * r < dv) w[r] = ld16<vec8>(Bh + c0 + (int64_t)(grp + 64 * r) * sVr);
    }
  };
  load_w();
  const int L = kv_lens ? kv_lens[b] : kv_len;
  const int nlive = live_splits(L, effective_splits(L, asked_splits(num_kv_splits, b, max_splits, split_cap), split_cap_in_force(split_cap, split_plan)), max_splits);
  const PartialRows rows = partial_rows(b, hq, max_splits, num_kv_splits, split_plan);
  float* head_lse = merged + hpw * dv;            // TAIL: [hpw][3] prefix log-sum-exp, the tail's maximum and sum; then [hpw][MERGE_CB] its rows
  if constexpr (TAIL) {
    float* rows_t = head_lse + 3 * hpw;
    for (int i = tid; i < hpw * MERGE_CB; i += MERGE_UP_T) {
      const int gi = i / MERGE_CB, c = c0 + i % MERGE_CB;
      if (c < d_out) {
        const int64_t row = ((int64_t)b * hq + hfirst + gi) * tail.splits;
        const MergeAcc<1> a = merge_fold<1>(tail.lse + row, tail.partial + row * d_out + c, d_out, 0, 1, tail.splits);
        rows_t[i] = a.acc[0];
        if (c == c0) { head_lse[3 * gi + 1] = a.m; head_lse[3 * gi + 2] = a.l; }
      }
    }
  }
  auto merge_packet = [&](int gi, int c, auto tag) {
    constexpr int P = decltype(tag)::value;
    const int64_t row = rows.base + (int64_t)(hfirst + gi) * rows.per_head;
    // a single row's weight is 1 whatever its log-sum-exp
    const MergeAcc<P> a = merge_fold<P>(max_splits == 1 && !lse_out && !TAIL ? nullptr : lse + row, partial + row * dv + c, dv, 0, 1, nlive);
    if (TAIL && c == 0) head_lse[3 * gi] = a.m + __logf(a.l);
    const float inv = nlive > 0 ? 1.f / a.l : 0.f;
#pragma unroll
    for (int e = 0; e < P; ++e) merged[gi * dv + c + e] = a.acc[e] * inv;
    if (lse_out && c == 0 && blockIdx.z == 0) lse_out[b * sLb + (hfirst + gi) * sLh] = a.m + __logf(a.l);
  };
  auto merge_shared = [&](auto tag) {             // MANY_SPREAD: head hfirst, its splits dealt out among MERGE_UP_T / (dv / P) groups
    constexpr int P = decltype(tag)::value;
    float* red = merged + dv;
    float* ml = red + MERGE_UP_T * P;
    const int lanes = dv / P, ngrp = MERGE_UP_T / lanes, sg = tid / lanes, c = (tid % lanes) * P;
    const int64_t row = rows.base + (int64_t)hfirst * rows.per_head;
    if (sg < ngrp) {
      const MergeAcc<P> a = merge_fold<P>(lse + row, partial + row * dv + c, dv, sg, ngrp, nlive);
#pragma unroll
      for (int e = 0; e < P; ++e) red[tid * P + e] = a.acc[e];
      ml[2 * tid] = a.m;
      ml[2 * tid + 1] = a.l;
    }
    __syncthreads();
    if (sg) return;
    float M = ml[2 * tid];
    for (int g = 1; g < ngrp; ++g) M = fmaxf(M, ml[2 * (g * lanes + tid)]);
    float l = 0.f, acc[P];
#pragma unroll
    for (int e = 0; e < P; ++e) acc[e] = 0.f;
    for (int g = 0; g < ngrp; ++g) {
      const int t = g * lanes + tid;
      const float x = ml[2 * t] == NEG_INF ? 0.f : __expf(ml[2 * t] - M);
      l += x * ml[2 * t + 1];
#pragma unroll
      for (int e = 0; e < P; ++e) acc[e] += x * red[t * P + e];
    }
    const float inv = nlive > 0 ? 1.f / l : 0.f;
#pragma unroll
    for (int e = 0; e < P; ++e) merged[c + e] = acc[e] * inv;
    if (lse_out && c == 0 && blockIdx.z == 0) lse_out[b * sLb + hfirst * sLh] = M + __logf(l);
  };
  const bool vec = (dv & 3) == 0 && (reinterpret_cast<uintptr_t>(partial) & 15) == 0;
  if constexpr (MANY == MANY_SPREAD) {
    if (vec) merge_shared(std::integral_constant<int, 4>());
    else merge_shared(std::integral_constant<int, 1>());
  } else if (vec) {
    const int ppr = dv >> 2;
    for (int i = tid; i < hpw * ppr; i += MERGE_UP_T) merge_packet(i / ppr, (i % ppr) * 4, std::integral_constant<int, 4>());
  } else {
    for (int i = tid; i < hpw * dv; i += MERGE_UP_T) merge_packet(i / dv, i % dv, std::integral_constant<int, 1>());
  }
  __syncthreads();
  for (;;) {                                      // this workgroup's column blocks
    for (int g0 = 0; g0 < hpw; g0 += HP) {
      float acc[8 * HP];                            // [heads][8 columns]
#pragma unroll
      for (int i = 0; i < 8 * HP; ++i) acc[i] = 0.f;
#pragma unroll
      for (int r = 0; r < RPT; ++r) {
        const int rho = grp + 64 * r;
#pragma unroll
        for (int gi = 0; gi < HP; ++gi) {
          const float m = g0 + gi < hpw && rho < dv ? merged[(g0 + gi) * dv + rho] : 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[gi * 8 + e] += m * to_f32(w[r][e]);
        }
      }
      // halving exchanges over the 16 lanes that share a column block: partner 15 - l, then 7 - l, 3 - l, 1 - l of the shrinking
      // group; the lane with the bit set keeps the upper half
#define XKV_HALVE(N, BIT, CTRL)                                                                                               \
    {                                                                                                                         \
      const bool up = lane & BIT;                                                                                             \
      _Pragma("unroll") for (int i = 0; i < N; ++i) {                                                                         \
        const float give = up ? acc[i] : acc[N + i], keep = up ? acc[N + i] : acc[i];                                         \
        acc[i] = keep + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, give), CTRL, 0xf, 0xf, false)); \
      }                                                                                                                       \
      }
      XKV_HALVE(4 * HP, 8, 0x140)   // row_mirror
      XKV_HALVE(2 * HP, 4, 0x141)   // row_half_mirror
      XKV_HALVE(HP, 2, 0x1B)        // quad_perm [3,2,1,0]
      const int idx = (lane & 8 ? 4 * HP : 0) + (lane & 4 ? 2 * HP : 0) + (lane & 2 ? HP : 0) + (lane & 1 ? HP / 2 : 0);   // this lane's sums
      if constexpr (HP == 4) {
        XKV_HALVE(2, 1, 0xB1)       // quad_perm [1,0,3,2]
#pragma unroll
        for (int i = 0; i < 2; ++i) tot[wave >> 1][((idx + i) >> 3) * MERGE_CB + cb * 8 + ((idx + i) & 7)] = acc[i];
      } else {
        const float sum = acc[0] + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, acc[0]), 0xB1, 0xf, 0xf, false));
        if (!(lane & 1)) tot[wave >> 1][cb * 8 + idx] = sum;
      }
#undef XKV_HALVE
      __syncthreads();
      if (tid < HP * MERGE_CB) {
        const int gi = tid / MERGE_CB, c = c0 + tid % MERGE_CB;
        if (g0 + gi < hpw && c < d_out) {
          float v = tot[0][tid] + tot[1][tid] + tot[2][tid] + tot[3][tid];
          if constexpr (TAIL) {
            const float *h = head_lse + 3 * (g0 + gi), M = fmaxf(h[0], h[1]), wp = __expf(h[0] - M), wt = __expf(h[1] - M);
            v = (v * wp + head_lse[3 * hpw + (g0 + gi) * MERGE_CB + c - c0] * wt) / (wp + h[2] * wt);
          }
          out[b * sOb + (hfirst + g0 + gi) * sOh + c] = (O)v;
        }
      }
      __syncthreads();            // tot is reused by the next four heads, or the next columns
    }
    if constexpr (MANY == ONE_PASS || MANY == ONE_HEAD) return;
    c0 += gridDim.z * MERGE_CB;
    if (c0 >= d_out) return;
    load_w();
  }
}

template <typename O>
static int launch_rope(void* s, void* c, const float* inv, int64_t seqlen, int64_t start, int half_dim,
                       hipStream_t st) {
  int64_t n = seqlen * half_dim;
  rope_table_kernel<O><<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st>>>((O*)s, (O*)c, inv, seqlen, start,
                                                                               half_dim);
  return launch_status();
}

template <typename O, typename TB>
static int launch_merge(const float* partial, const float* lse, void* out, const void* vB, int64_t sVb, int64_t sVh,
                        int64_t sVr, int d_out, const int32_t* ns, const int32_t* kl, int batch, int hq, int hkv,
                        int kv_len, int max_splits, int dv, int64_t sOb, int64_t sOh, float* lse_out, int64_t sLb, int64_t sLh,
                        int split_cap, const int32_t* split_plan, const MergeTail& tail, hipStream_t st) {
  // splits one sequence may have (a packed plan's max_splits counts the jobs of the whole batch)
  const int seq_splits = packed_rows(ns, split_plan) ? std::min(max_splits, cdiv(kv_len, split_cap)) : max_splits;
  // what one head takes of the LDS was bounded when the weights of all its splits were held there; the bound stays part of the
  // interface (a split count this large is refused before any launch)
  if ((size_t)(dv + seq_splits) * sizeof(float) > 24 * 1024) return XKV_EUNSUPPORTED;
  if (!vB) {
    // few splits: a head's whole row per workgroup; more: narrower feature blocks, so that a thread folds few splits, until the
    // grid fills the chip four times over
    const bool vec = dv % 4 == 0 && (reinterpret_cast<uintptr_t>(partial) & 15) == 0;
    int chunk = vec ? 1024 : 256;
    while (chunk / 2 >= dv || (chunk > 64 && (int64_t)seq_splits * chunk > (vec ? 8192 : 2048) &&
                               (int64_t)hq * batch * cdiv(dv, chunk) < 1024))
      chunk /= 2;
    const dim3 grid(hq, batch, cdiv(dv, chunk));
    if (vec)
      merge_rows_kernel<O, 4><<<grid, dim3(256), 0, st>>>(partial, lse, (O*)out, ns, kl, hq, kv_len, max_splits, dv, chunk, sOb, sOh,
                                                          lse_out, sLb, sLh, split_cap, split_plan);
    else
      merge_rows_kernel<O, 1><<<grid, dim3(256), 0, st>>>(partial, lse, (O*)out, ns, kl, hq, kv_len, max_splits, dv, chunk, sOb, sOh,
                                                          lse_out, sLb, sLh, split_cap, split_plan);
    return launch_status();
  }
  // Many splits (a caller with scratch to spare merges the rows first, as the wrappers do): where the heads fill the chip a workgroup
  // folds once for several column blocks; where they do not even with a workgroup per block, a workgroup takes one head and deals
  // its splits out among groups of threads, as it does wherever that is the faster (merge_rule.h).
  int hpw = merge_heads(hq, hkv, dv, batch, d_out);
  int z = cdiv(d_out, MERGE_CB);
  const bool many = tail.splits ? merge_tail_rows_first(seq_splits, hq, hkv, dv) : seq_splits > 1 && (int64_t)seq_splits * hpw * dv > MERGE_FLOATS;
  const bool spread = !tail.splits && (merge_spread(seq_splits, hq, batch, dv, d_out) || (many && (int64_t)(hq / hpw) * batch * z < 256));
  const bool head = !many && !spread && merge_one_head(hq, batch, d_out);
  if (spread || head) hpw = 1;
  if (many || spread) z = (int)std::min<int64_t>(z, cdiv(256, std::min<int64_t>(256, (int64_t)(hq / hpw) * batch)));
  const dim3 grid(hq / hpw, batch, z);
  const size_t shm = ((size_t)hpw * dv + (spread ? MERGE_UP_T * 6 : 0) + (tail.splits ? hpw * (MERGE_CB + 3) : 0)) * sizeof(float);
#define XKV_MERGE_UP_TAIL(RPT, MANY, TAIL)                                                                                           \
  merge_up_kernel<O, TB, RPT, MANY, TAIL><<<grid, dim3(MERGE_UP_T), shm, st>>>(partial, lse, (O*)out, (const TB*)vB, sVb, sVh, sVr, d_out, ns, kl, \
                                                         hq, hkv, kv_len, max_splits, dv, sOb, sOh, hpw, lse_out, sLb, sLh, split_cap, split_plan, tail)
#define XKV_MERGE_UP(RPT, MANY) XKV_MERGE_UP_TAIL(RPT, MANY, false)
  if (tail.splits) {
    if (many) return XKV_EUNSUPPORTED;   // the caller merges the rows first
    if constexpr (std::is_same<O, TB>::value) {
      if (head) { if (dv <= 256) XKV_MERGE_UP_TAIL(4, ONE_HEAD, true); else XKV_MERGE_UP_TAIL(8, ONE_HEAD, true); }
      else { if (dv <= 256) XKV_MERGE_UP_TAIL(4, ONE_PASS, true); else XKV_MERGE_UP_TAIL(8, ONE_PASS, true); }
      return launch_status();
    }
    return XKV_EDTYPE;
  }
  if (dv <= 256) { if (spread) XKV_MERGE_UP(4, MANY_SPREAD); else if (many) XKV_MERGE_UP(4, MANY_LOOP); else if (head) XKV_MERGE_UP(4, ONE_HEAD); else XKV_MERGE_UP(4, ONE_PASS); }
  else { if (spread) XKV_MERGE_UP(8, MANY_SPREAD); else if (many) XKV_MERGE_UP(8, MANY_LOOP); else if (head) XKV_MERGE_UP(8, ONE_HEAD); else XKV_MERGE_UP(8, ONE_PASS); }
#undef XKV_MERGE_UP
#undef XKV_MERGE_UP_TAIL
  return launch_status();
}

// plan[0]: smallest multiple of 32 >= floor_tokens with sum_b ceil(len_b / cap) <= target_jobs.  Then the job list: sequence b
// has n_b = effective_splits(len_b, num_splits[b], cap) splits of which the live ones are a prefix; whole splits first
// (sequence-major), every sequence's last live split - the short one - after them.
// One workgroup in front of the scan, so its latency is the call's: the answer lies between total / target (no split is
// longer) and total / (target - batch) (every sequence wastes less than one split), a range of a few dozen caps that 32 groups of
// 32 threads test at once; and a job finds its sequence by bisection in the prefix sums instead of one thread writing all jobs
// of its sequence.  By trace, 32 sequences of 1K .. 128K tokens: 4.9 us, 8 sequences: 3.9; a 256-ary search over all
// caps with one thread per candidate and per sequence: 9.4 and 6.3.
constexpr int PLAN_T = 512, PLAN_W = PLAN_T / 64;
// ceil(n / d) for n >= 0, d > 0: a float quotient, corrected by its remainder, a third of the
// instructions of an integer division
__device__ __forceinline__ int plan_cdiv(int n, int d) {
  int q = (int)((float)n * __builtin_amdgcn_rcpf((float)d));
  int r = n - q * d;
  while (r < 0) { --q; r += d; }
  while (r >= d) { ++q; r -= d; }
  return q + (r > 0 ? 1 : 0);
}
__global__ __launch_bounds__(PLAN_T) void plan_splits_kernel(const int32_t* __restrict__ kv_lens, const int32_t* __restrict__ num_splits,
                                                             int batch, int max_splits, int floor_tokens, int target_jobs,
                                                             int32_t* __restrict__ plan) {
  __shared__ int lens[PLAN_T], pre[PLAN_T + 1];
  __shared__ float redf[PLAN_W];
  __shared__ int redm[PLAN_W], red1[PLAN_W], fit[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // longest length, total length (a float sum: it only bounds the search); the first PLAN_T lengths stay in the LDS
  int longest = 0;
  float total = 0.f;
  for (int b = tid; b < batch; b += PLAN_T) {
    const int L = kv_lens[b] > 0 ? kv_lens[b] : 0;
    if (b < PLAN_T) lens[b] = L;
    longest = L > longest ? L : longest;
    total += (float)L;
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int w = __shfl_xor(longest, o);
    longest = w > longest ? w : longest;
    total += __shfl_xor(total, o);
  }
  if (lane == 0) { redm[wave] = longest; redf[wave] = total; }
  if (tid == 0) fit[0] = fit[1] = PLAN_T;
  __syncthreads();
  longest = 0;
  total = 0.f;
#pragma unroll
  for (int i = 0; i < PLAN_W; ++i) { longest = redm[i] > longest ? redm[i] : longest; total += redf[i]; }
  auto len_of = [&](int b) { const int L = b < PLAN_T ? lens[b] : kv_lens[b]; return L > 0 ? L : 0; };
  // caps in units of 32 tokens: the answer is in [lo, hi]; if even one job per sequence is too many it is the longest length
  int lo = cdiv(floor_tokens > 32 ? floor_tokens : 32, 32), hi = cdiv(longest > 32 ? longest : 32, 32);
  if (hi < lo) hi = lo;
  const int floor_units = lo;
  {
    // total / cap <= jobs from below, jobs < total / cap + batch from above; 0.1 % of slack covers the float sum
    const int least = (int)fminf(total * 0.999f / ((float)target_jobs * 32.f), (float)hi);
    if (least > lo) lo = least;
    if (target_jobs > batch) {
      const int most = (int)fminf(total * 1.001f / ((float)(target_jobs - batch) * 32.f), (float)hi) + 1;
      if (most < hi) hi = most > floor_units ? most : floor_units;
      if (hi < lo) hi = lo;
    }
  }
  const int cand = tid >> 5, sub = tid & 31;
  for (int round = 0; lo < hi; ++round) {
    const int stride = cdiv(hi - lo + 1, PLAN_T / 32);   // candidate i tests the last cap of its block; the first that fits wins
    const int first = lo + cand * stride;
    int c = first + stride - 1;
    c = c < hi ? c : hi;
    int jobs = 0;
    if (first <= hi)
      for (int b = sub; b < batch; b += 32) jobs += plan_cdiv(len_of(b), c * 32);
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) jobs += __shfl_xor(jobs, o);
    if (sub == 0 && first <= hi && jobs <= target_jobs) atomicMin(&fit[round & 1], cand);
    __syncthreads();
    const int f = fit[round & 1];
    __syncthreads();
    if (tid == 0) fit[round & 1] = PLAN_T;               // next used two rounds on, behind the next round's barriers
    if (f == PLAN_T) { lo = hi; break; }
    lo += f * stride;
    hi = lo + stride - 1 < hi ? lo + stride - 1 : hi;
  }
  const int cap = lo * 32;
  // live splits of a sequence, in the arithmetic of split_bounds
  auto live_of = [&](int b) {
    const int L = len_of(b);
    if (L <= 0) return 0;
    const int asked = asked_splits(num_splits, b, max_splits, cap), fit_n = plan_cdiv(L, cap), n = fit_n > asked ? fit_n : asked;
    const int per = (plan_cdiv(L, n) + MIN_BLOCK_KV - 1) / MIN_BLOCK_KV * MIN_BLOCK_KV;
    const int live = plan_cdiv(L, per);
    return live < max_splits ? live : max_splits;
  };
  // whole splits of every sequence first, then the last ones: `whole` is where the second list starts
  int whole = 0;
  if (batch > PLAN_T) {                    // several chunks of sequences: the length of the first list is needed up front
    int n = 0;
    for (int b = tid; b < batch; b += PLAN_T) { const int l = live_of(b); n += l > 0 ? l - 1 : 0; }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) n += __shfl_xor(n, o);
    __syncthreads();
    if (lane == 0) redm[wave] = n;
    __syncthreads();
    for (int i = 0; i < PLAN_W; ++i) whole += redm[i];
  }
  int done = 0, last = 0;
  for (int b0 = 0; b0 < batch; b0 += PLAN_T) {
    const int b = b0 + tid, live = b < batch ? live_of(b) : 0;
    const int m0 = live > 0 ? live - 1 : 0, m1 = live > 0 ? 1 : 0;
    int i0 = m0, i1 = m1;                  // inclusive scans within the wave, then across the waves
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int w0 = __shfl_up(i0, o), w1 = __shfl_up(i1, o);
      if (lane >= o) { i0 += w0; i1 += w1; }
    }
    __syncthreads();
    if (lane == 63) { redm[wave] = i0; red1[wave] = i1; }
    __syncthreads();
    int all0 = 0, all1 = 0;
#pragma unroll
    for (int i = 0; i < PLAN_W; ++i) {
      if (i == wave) { i0 += all0; i1 += all1; }
      all0 += redm[i];
      all1 += red1[i];
    }
    pre[tid + 1] = i0;
    if (tid == 0) pre[0] = 0;
    if (batch <= PLAN_T) whole = all0;
    __syncthreads();
    for (int j = tid; j < all0; j += PLAN_T) {   // the sequence of job j: the last one whose jobs start at or before j
      int l = 0, r = PLAN_T - 1;
      while (l < r) {
        const int m = (l + r + 1) >> 1;
        if (pre[m] <= j) l = m; else r = m - 1;
      }
      plan[2 + 2 * (done + j)] = b0 + l;
      plan[3 + 2 * (done + j)] = j - pre[l];
    }
    if (m1) {
      plan[2 + 2 * (whole + last + i1 - 1)] = b;
      plan[3 + 2 * (whole + last + i1 - 1)] = live - 1;
    }
    // a packed plan: the partial rows of the sequences lie behind each other
    if (!num_splits && b < batch) plan[2 + 2 * (int64_t)max_splits + b] = done + last + (i0 - m0) + (i1 - m1);
    done += all0;
    last += all1;
  }
  if (tid == 0) {
    plan[0] = cap;
    plan[1] = done + last;
    if (!num_splits) plan[2 + 2 * (int64_t)max_splits + batch] = done + last;
  }
}

}  // namespace xkv

using namespace xkv;

extern "C" int xkv_plan_splits(const int32_t* kv_lens, const int32_t* num_kv_splits, int batch, int max_splits, int floor_tokens,
                               int target_jobs, int32_t* plan, void* stream) {
  if (!kv_lens || !plan || batch <= 0 || max_splits <= 0 || floor_tokens <= 0 || target_jobs <= 0) return XKV_EINVAL;
  // without an array of counts the caps alone make the jobs: at most target_jobs, or one a sequence
  if (!num_kv_splits && max_splits < std::max(batch, target_jobs)) return XKV_EINVAL;
  plan_splits_kernel<<<dim3(1), dim3(PLAN_T), 0, (hipStream_t)stream>>>(kv_lens, num_kv_splits, batch, max_splits, floor_tokens,
                                                                     target_jobs, plan);
  return launch_status();
}

extern "C" int xkv_abi_version(void) { return XKV_ABI_VERSION; }

extern "C" const char* xkv_error_string(int code) {
  switch (code) {
    case XKV_OK: return "ok";
    case XKV_EINVAL: return "invalid argument (null pointer or non-positive size)";
    case XKV_EUNSUPPORTED: return "shape outside the built envelope";
    case XKV_EALIGN: return "pointer or stride not 16-byte aligned";
    case XKV_EDTYPE: return "unsupported dtype code";
    case XKV_ESCRATCH: return "the call needs more scratch than the library's static device array holds";
    case XKV_ETOOLCHAIN: return "a kernel that tracks its own loads was built with register spills: rebuild with the validated compiler";
    default: return code > 0 ? hipGetErrorString((hipError_t)code) : "unknown xkv error";
  }
}

extern "C" int xkv_rope_table(void* sin_out, void* cos_out, const float* inv_freq, int64_t seqlen, int64_t start,
                              int half_dim, int out_dtype, void* stream) {
  if (!sin_out || !cos_out || !inv_freq || seqlen < 0 || half_dim <= 0) return XKV_EINVAL;
  if (seqlen == 0) return XKV_OK;
  hipStream_t st = (hipStream_t)stream;
  switch (out_dtype) {
    case XKV_F32: return launch_rope<float>(sin_out, cos_out, inv_freq, seqlen, start, half_dim, st);
    case XKV_F16: return launch_rope<_Float16>(sin_out, cos_out, inv_freq, seqlen, start, half_dim, st);
    case XKV_BF16: return launch_rope<__bf16>(sin_out, cos_out, inv_freq, seqlen, start, half_dim, st);
    default: return XKV_EDTYPE;
  }
}

template <typename T>
static int launch_rope_apply(const void* x, void* out, const float* inv_freq, const int64_t* positions, int64_t pos0,
                             int batch, int rows, int heads, int dim, int64_t sxb, int64_t sxr, int64_t sxh, int64_t sob,
                             int64_t sor, int64_t soh, hipStream_t st) {
  const int64_t total = (int64_t)batch * rows * heads * (dim / 2);
  const int64_t blocks = (total + 255) / 256;
  if (blocks > 0x7fffffff) return XKV_EUNSUPPORTED;
  rope_apply_kernel<T><<<dim3((unsigned)blocks), dim3(256), 0, st>>>((const T*)x, (T*)out, inv_freq, positions, pos0, total, rows,
                                                                      heads, dim / 2, sxb, sxr, sxh, sob, sor, soh);
  return launch_status();
}

extern "C" int xkv_rope_apply(const void* x, void* out, const float* inv_freq, const int64_t* positions, int64_t pos0,
                              int batch, int rows, int heads, int dim, int64_t sxb, int64_t sxr, int64_t sxh,
                              int64_t sob, int64_t sor, int64_t soh, int dtype, void* stream) {
  if (!x || !out || !inv_freq || batch < 0 || rows < 0 || heads <= 0 || dim <= 0) return XKV_EINVAL;
  if (dim % 2) return XKV_EUNSUPPORTED;
  if (batch == 0 || rows == 0) return XKV_OK;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case XKV_F32: return launch_rope_apply<float>(x, out, inv_freq, positions, pos0, batch, rows, heads, dim, sxb, sxr, sxh, sob, sor, soh, st);
    case XKV_F16: return launch_rope_apply<_Float16>(x, out, inv_freq, positions, pos0, batch, rows, heads, dim, sxb, sxr, sxh, sob, sor, soh, st);
    case XKV_BF16: return launch_rope_apply<__bf16>(x, out, inv_freq, positions, pos0, batch, rows, heads, dim, sxb, sxr, sxh, sob, sor, soh, st);
    default: return XKV_EDTYPE;
  }
}

extern "C" int xkv_absorb_q(const void* q, const void* B, void* qt_hi, void* qt_lo, int batch, int hq, int hkv, int d,
                            int rank, int64_t sBb, int64_t sBh, int64_t sBr, int dtype, void* stream) {
  if (!q || !B || !qt_hi || batch <= 0 || hq <= 0 || hkv <= 0 || d <= 0 || rank <= 0) return XKV_EINVAL;
  if (hq % hkv || hq / hkv > 32 || d > 512 || d % 8) return XKV_EUNSUPPORTED;
  if (sBr % 8 || sBh % 8 || sBb % 8 || ((uintptr_t)B & 15)) return XKV_EALIGN;
  hipStream_t st = (hipStream_t)stream;
  if (dtype != XKV_BF16 && dtype != XKV_F16) return XKV_EDTYPE;
  const dim3 block(256);
  const int nhb = (hq / hkv + 15) / 16;   // blocks of 16 query heads per kv head
  // the MFMA form reads 16-byte packets of q: a query buffer that is not aligned takes the scalar form, as does a head_dim
  // that is not a whole number of 32-feature k-steps; beyond eight k-steps (d 256) the waves of a workgroup share them
#define XKV_ABSORB(T)                                                                                                          \
  if (d % 32 == 0 && ((uintptr_t)q & 15) == 0 && d > 256)                                                                      \
    absorb_q_mfma_kernel<T, true><<<dim3(hkv * nhb, batch, (rank + 15) / 16), block, 0, st>>>((const T*)q, (const T*)B, (T*)qt_hi, \
                                                                                 (T*)qt_lo, hq, hkv, d, rank, sBb, sBh, sBr);  \
  else if (d % 32 == 0 && ((uintptr_t)q & 15) == 0)                                                                            \
    absorb_q_mfma_kernel<T, false><<<dim3(hkv * nhb, batch, (rank + 63) / 64), block, 0, st>>>((const T*)q, (const T*)B, (T*)qt_hi, \
                                                                                 (T*)qt_lo, hq, hkv, d, rank, sBb, sBh, sBr);  \
  else                                                                                                                         \
    absorb_q_kernel<T><<<dim3(hkv, batch, (rank + 255) / 256), block, 0, st>>>((const T*)q, (const T*)B, (T*)qt_hi, (T*)qt_lo, \
                                                                                 hq, hkv, d, rank, sBb, sBh, sBr);
  if (dtype == XKV_BF16) { XKV_ABSORB(__bf16) } else { XKV_ABSORB(_Float16) }
#undef XKV_ABSORB
  return launch_status();
}

extern "C" int xkv_blockdiag_q(const void* q, void* out, int batch, int hq, int hkv, int d, int dtype, void* stream) {
  if (!q || !out || batch <= 0 || hq <= 0 || hkv <= 0 || d <= 0) return XKV_EINVAL;
  if (hq % hkv || d % 8) return XKV_EUNSUPPORTED;
  if (((uintptr_t)q & 15) || ((uintptr_t)out & 15)) return XKV_EALIGN;
  const int64_t total8 = (int64_t)batch * hq * hkv * d / 8;
  const dim3 grid((unsigned)((total8 + 255) / 256)), block(256);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == XKV_BF16) blockdiag_q_kernel<__bf16><<<grid, block, 0, st>>>((const __bf16*)q, (__bf16*)out, hq, hkv, d, total8);
  else if (dtype == XKV_F16) blockdiag_q_kernel<_Float16><<<grid, block, 0, st>>>((const _Float16*)q, (_Float16*)out, hq, hkv, d, total8);
  else return XKV_EDTYPE;
  return launch_status();
}

extern "C" int xkv_merge_stage2(const float* partial, const float* lse, void* out, const void* vB, int64_t sVb,
                                int64_t sVh, int64_t sVr, int d_out, int vB_dtype, const int32_t* ns,
                                const int32_t* kl, int batch, int hq, int hkv, int kv_len, int max_splits,
                                int split_cap_tokens, const int32_t* split_plan, int dv, int64_t sOb, int64_t sOh, int out_dtype, float* lse_out,
                                int64_t sLb, int64_t sLh, void* stream) {
  if (!partial || !lse || !out || batch <= 0 || hq <= 0 || hkv <= 0 || max_splits <= 0 || dv <= 0)
    return XKV_EINVAL;
  if (!cap_fits(ns, batch, kv_len, max_splits, split_cap_tokens, split_plan)) return XKV_EINVAL;
  if (hq % hkv || hq / hkv > 32 || dv > 512) return XKV_EUNSUPPORTED;
  if (vB && (d_out <= 0 || d_out > 512 || d_out % 8)) return XKV_EUNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
#define XKV_MERGE(O, TB) \
  return launch_merge<O, TB>(partial, lse, out, vB, sVb, sVh, sVr, d_out, ns, kl, batch, hq, hkv, kv_len, max_splits, dv, sOb, sOh, lse_out, sLb, sLh, split_cap_tokens, split_plan, MergeTail{nullptr, nullptr, 0}, st)
  const int bt = vB ? vB_dtype : XKV_BF16;
  if (bt != XKV_BF16 && bt != XKV_F16) return XKV_EDTYPE;
  switch (out_dtype) {
    case XKV_F32: if (bt == XKV_BF16) XKV_MERGE(float, __bf16); else XKV_MERGE(float, _Float16);
    case XKV_F16: if (bt == XKV_BF16) XKV_MERGE(_Float16, __bf16); else XKV_MERGE(_Float16, _Float16);
    case XKV_BF16: if (bt == XKV_BF16) XKV_MERGE(__bf16, __bf16); else XKV_MERGE(__bf16, _Float16);
    default: return XKV_EDTYPE;
  }
#undef XKV_MERGE
}

extern "C" int xkv_absorb_q_tail(const void* q, const void* B, void* qt_hi, void* qt_lo, int batch, int hq, int hkv, int d, int rank,
                                 int64_t sBb, int64_t sBh, int64_t sBr, xkv_kv_operand k_tail, xkv_kv_operand v_tail, int tail_len,
                                 int tail_splits, float* tail_partial, float* tail_lse, float sm_scale, float logit_cap, int dtype,
                                 void* stream) {
  if (!q || !B || !qt_hi || !k_tail.ptr || !v_tail.ptr || !tail_partial || !tail_lse || batch <= 0 || hq <= 0 || hkv <= 0 || d <= 0 ||
      rank <= 0 || tail_len <= 0 || tail_splits <= 0)
    return XKV_EINVAL;
  if (hq % hkv || hq / hkv > 32 || d > 512 || d % 32 || k_tail.dim != d || v_tail.dim <= 0 || v_tail.dim % 64 || v_tail.dim > 512)
    return XKV_EUNSUPPORTED;
  const int blocks = cdiv(tail_len, 32), tiles = cdiv(blocks, tail_splits);
  if (cdiv(blocks, tiles) != tail_splits) return XKV_EINVAL;   // every split of the tail holds tokens
  if ((sBr | sBh | sBb | k_tail.stride_b | k_tail.stride_l | v_tail.stride_b | v_tail.stride_l) & 7 ||
      ((uintptr_t)B | (uintptr_t)q | (uintptr_t)k_tail.ptr | (uintptr_t)v_tail.ptr | (uintptr_t)tail_partial) & 15)
    return XKV_EALIGN;
  if (dtype != XKV_BF16 && dtype != XKV_F16) return XKV_EDTYPE;
  TailParams t;
  t.k = k_tail.ptr; t.v = v_tail.ptr;
  t.sKb = k_tail.stride_b; t.sKl = k_tail.stride_l; t.sVb = v_tail.stride_b; t.sVl = v_tail.stride_l;
  t.partial = tail_partial; t.lse = tail_lse;
  t.len = tail_len; t.splits = tail_splits; t.tiles = tiles; t.dv = v_tail.dim;
  t.groups = cdiv(hq, 32);
  while (hq % t.groups) ++t.groups;
  t.sm_scale = sm_scale; t.logit_cap = logit_cap;
  const bool ksplit = d > 256;
  t.head_blocks = hkv * ((hq / hkv + 15) / 16);
  t.rank_blocks = ksplit ? cdiv(rank, 16) : cdiv(rank, 64);
  const int64_t absorbing = (int64_t)t.head_blocks * t.rank_blocks * batch, grid = absorbing + (int64_t)batch * t.groups * tail_splits;
  if (grid > 0x7fffffff) return XKV_EUNSUPPORTED;
  t.absorbing = (int)absorbing;
  const size_t shm = (size_t)32 * (t.dv + 8) * 2;
  hipStream_t st = (hipStream_t)stream;
#define XKV_ABSORB_TAIL(T, KS) \
  absorb_tail_kernel<T, KS><<<dim3((unsigned)grid), dim3(256), shm, st>>>((const T*)q, (const T*)B, (T*)qt_hi, (T*)qt_lo, hq, hkv, d, rank, sBb, sBh, sBr, t)
  if (dtype == XKV_BF16) { if (ksplit) XKV_ABSORB_TAIL(__bf16, true); else XKV_ABSORB_TAIL(__bf16, false); }
  else { if (ksplit) XKV_ABSORB_TAIL(_Float16, true); else XKV_ABSORB_TAIL(_Float16, false); }
#undef XKV_ABSORB_TAIL
  return launch_status();
}

extern "C" int xkv_merge_stage2_tail(const float* partial, const float* lse, void* out, const void* vB, int64_t sVb, int64_t sVh,
                                     int64_t sVr, int d_out, int dtype, int batch, int hq, int hkv, int kv_len, int max_splits, int dv,
                                     const float* tail_partial, const float* tail_lse, int tail_splits, int64_t sOb, int64_t sOh,
                                     void* stream) {
  if (!partial || !lse || !out || !vB || !tail_partial || !tail_lse || batch <= 0 || hq <= 0 || hkv <= 0 || max_splits <= 0 || dv <= 0 ||
      kv_len <= 0 || tail_splits <= 0)
    return XKV_EINVAL;
  if (hq % hkv || hq / hkv > 32 || dv > 512 || d_out <= 0 || d_out > 512 || d_out % 8) return XKV_EUNSUPPORTED;
  const MergeTail tail{tail_partial, tail_lse, tail_splits};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == XKV_BF16)
    return launch_merge<__bf16, __bf16>(partial, lse, out, vB, sVb, sVh, sVr, d_out, nullptr, nullptr, batch, hq, hkv, kv_len, max_splits, dv,
                                        sOb, sOh, nullptr, 0, 0, 0, nullptr, tail, st);
  if (dtype == XKV_F16)
    return launch_merge<_Float16, _Float16>(partial, lse, out, vB, sVb, sVh, sVr, d_out, nullptr, nullptr, batch, hq, hkv, kv_len, max_splits,
                                            dv, sOb, sOh, nullptr, 0, 0, 0, nullptr, tail, st);
  return XKV_EDTYPE;
}
