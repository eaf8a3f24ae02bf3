// Scores of rotated reconstructed keys at ranks up to 192:  K = kA @ kB[kh]  ->  rotate-half RoPE  ->  q . K'  ->  [batch, hq, kv_len].
//
// At these ranks a kv head's whole factor (rank x 128, 48 KB at 192) fits the accumulation registers of ONE wave, so a wave
// rebuilds 16 tokens by itself: no partial scores to add up, no barrier and no LDS tile.  In the workgroup-wide form (four
// waves share a 32-token tile, two barriers and an LDS pass per tile) the period is latency - 1.4 us beside 0.15 us of MFMA - and
// does not fall with the rank; the waves here are independent.
//
// One workgroup owns one (batch, kv head, split); wave w takes the 16-token tiles w, w + 4, w + 8 ... of the split.  The token rows go from
// global memory straight into v_mfma_f32_16x16x32 as the B operand (a lane's packet is 8 consecutive ranks of one row),
// NBUF - 1 tiles ahead.  The 128 features are rebuilt 16 pairs (j, j + 64) at a time: while the matrix pipe works on one block of
// pairs the vector pipe rotates the one before, in fp32, and hands it, rounded to fp16, to the q-dot as its A operand.
//
// Measured at 131072 tokens, 8 kv heads: 61.4 us a launch at rank 192 (the workgroup-wide form 88), 58.2 at rank 128; 0.83 and 0.73 us
// per 64 tokens of a CU.  One wave per SIMD issues everything in order: of about 1900 cycles per tile at rank 192 the matrix pipe
// is busy for 832 and the rotation's vector instructions take 600.  Two waves per SIMD, each with half the features and the tile in
// the LDS, measured 64 - 67 us (twice the LDS reads, a barrier per step); coalesced rows through a wave-private LDS tile 64 - 68.
//
// cos / sin of a position: per-lane constants of the token's place in the wave's 64-token step times the step's base rotation.  The
// base lives one pair per lane, advanced by a constant rotation, re-seeded with a range-reduced sincosf every 16 steps and read back
// through a wave-private LDS row.
#include "recon_fast.h"
#include "xkv_common.h"
#include <type_traits>

namespace xkv {
namespace {

typedef short s16x4s __attribute__((ext_vector_type(4)));
typedef short s16x8s __attribute__((ext_vector_type(8)));
template <int V> using IC = std::integral_constant<int, V>;

constexpr int NBUF = 4;              // tiles of token rows in registers: one in use, three on the way
constexpr int STEP = 64;             // tokens a workgroup advances by: a tile of each wave
constexpr int BLD = 128 + 8;         // LDS row of the factor, elements
constexpr int SEED = 16;             // steps between range-reduced base angles

struct FactorOperand { const void* p; int64_t sb, sh, sr; };

template <typename T, int NKS>
__global__ __launch_bounds__(256, 1) void recon_scores_kernel(const FastParams p, const FactorOperand kB, const int vec_out) {
  typedef typename Elem<T>::vec8 vec8;
  typedef T vec4 __attribute__((ext_vector_type(4)));
  constexpr int RK = 32 * NKS;
  constexpr int TABLE = 4 * 16 * 64 * 2 * 4, FACTOR = RK * BLD * 2;
  // [wave][token of its tile][pair] cos, sin; then the factor
  __shared__ __attribute__((aligned(16))) unsigned char stage[TABLE > FACTOR ? TABLE : FACTOR];
  __shared__ __attribute__((aligned(16))) float base_lds[4][2][64 * 2];  // [wave][parity][pair] cos, sin of the step's first token
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, g4 = lane >> 4;

  const int wg = xcd_cluster_remap(blockIdx.x, p.hkv);   // the kv heads of one (sequence, split) stream the same rows: one L2
  if (wg >= p.total_wg) return;
  const int kh = wg % p.hkv;
  const int split = (wg / p.hkv) % p.max_splits;
  const int b = wg / (p.hkv * p.max_splits);
  const int L = p.kv_lens ? p.kv_lens[b] : p.kv_len;
  int start, end;
  split_bounds(L, asked_splits(p.num_splits, b, p.max_splits, 0), split, start, end);
  if (end <= start) return;
  const int G = p.hq / p.hkv, h0 = kh * G;
  const int last = end - 1;
  const int tok0 = start + 16 * wave;
  const int n = tok0 < end ? (end - tok0 + STEP - 1) / STEP : 0;

  // ---- token rows: lane (token n16, g4) holds ranks 32 ks + 8 g4 .. + 7; rows past the split repeat its last one -----------
  const T* Ab = reinterpret_cast<const T*>(p.kA) + b * p.sAb + 8 * g4;
  vec8 at[NBUF][NKS];
  auto load = [&](int i, auto buf_c) {
    int t = tok0 + i * STEP + n16;
    t = t < last ? t : last;
    const T* row = Ab + (int64_t)t * p.sAl;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) at[decltype(buf_c)::value][ks] = ld16<vec8>(row + 32 * ks);
  };
  load(0, IC<0>());
  load(1, IC<1>());
  load(2, IC<2>());

  // ---- the factor, through the LDS into accumulation registers: lane (feature n16, g4) holds 8 consecutive ranks ------------
  vec8 rows[2 * NKS];   // on the way while the angles are computed
  {
    const T* Bh = reinterpret_cast<const T*>(kB.p) + b * kB.sb + kh * kB.sh + (int64_t)(tid >> 4) * kB.sr + (tid & 15) * 8;
#pragma unroll
    for (int i = 0; i < 2 * NKS; ++i) rows[i] = ld16<vec8>(Bh + (int64_t)(16 * i) * kB.sr);
  }
  const float inv = p.inv_freq[lane];
  float c64, s64, cb = 1.f, sb = 0.f;
  sincosf((float)STEP * inv, &s64, &c64);
  float* table = reinterpret_cast<float*>(stage) + wave * (16 * 64 * 2);
  for (int o = 0; o < 16; ++o) {
    float s, c;
    sincosf((float)(16 * wave + o) * inv, &s, &c);
    *reinterpret_cast<float2*>(&table[(o * 64 + lane) * 2]) = make_float2(c, s);
  }
  // The table is written and read by this wave alone, whose LDS operations are carried out in order.  This lane's pairs are
  // j = 16 pb + 4 g4 + r, at token n16 of the tile.
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  f32x4 ci[4], si[4];
#pragma unroll
  for (int pb = 0; pb < 4; ++pb) {
    const float* src = table + (n16 * 64 + 16 * pb + 4 * g4) * 2;
    const f32x4 a = *reinterpret_cast<const f32x4*>(src), c = *reinterpret_cast<const f32x4*>(src + 4);
    ci[pb] = f32x4{a[0], a[2], c[0], c[2]};
    si[pb] = f32x4{a[1], a[3], c[1], c[3]};
  }
  __syncthreads();   // every wave has read its table
  T* factor = reinterpret_cast<T*>(stage);
#pragma unroll
  for (int i = 0; i < 2 * NKS; ++i) st16(factor + ((tid >> 4) + 16 * i) * BLD + (tid & 15) * 8, rows[i]);
  __syncthreads();
  vec8 breg[NKS][8];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
    for (int cbk = 0; cbk < 8; ++cbk) {
      const T* src = factor + (32 * ks + 8 * g4 + (n16 >> 2)) * BLD + 16 * cbk + 4 * (n16 & 3);
      s16x4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4s*)src);
      s16x4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4s*)(src + 4 * BLD));
      breg[ks][cbk] = __builtin_bit_cast(vec8, (s16x8s)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  // q operand: lane (head n16, g4) holds the same four pairs' low features and their partners
  sc_vec8 qop[4];
#pragma unroll
  for (int pb = 0; pb < 4; ++pb) {
    qop[pb] = sc_vec8{0, 0, 0, 0, 0, 0, 0, 0};
    if (n16 < G) {
      const T* qh = reinterpret_cast<const T*>(p.q) + ((int64_t)b * p.hq + h0 + n16) * 128 + 16 * pb + 4 * g4;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        qop[pb][e] = from_f32<sc_t>(to_f32(qh[e]));
        qop[pb][4 + e] = from_f32<sc_t>(to_f32(qh[64 + e]));
      }
    }
  }
  if (n == 0) return;

  f32x4 k[2][2];           // [parity of the block][low | partner features]
  f32x4 ba[2], bb[2];      // base rotation of the lane's pairs: cos, sin, cos, sin ...
  f32x4 s_cur = {0.f, 0.f, 0.f, 0.f}, s_prev;
  k[1][0] = k[1][1] = ba[1] = bb[1] = s_cur;

  auto rebuild = [&](auto buf_c, auto pb_c) {
    constexpr int B = decltype(buf_c)::value, PB = decltype(pb_c)::value;
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      lo = Elem<T>::mfma16(breg[ks][PB], at[B][ks], lo);
      hi = Elem<T>::mfma16(breg[ks][4 + PB], at[B][ks], hi);
    }
    k[PB & 1][0] = lo;
    k[PB & 1][1] = hi;
  };
  auto rotate_dot = [&](auto pb_c, f32x4 lo, f32x4 hi, f32x4 s) -> f32x4 {
    constexpr int PB = decltype(pb_c)::value;
    sc_vec8 kop;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const f32x4& base = r < 2 ? ba[PB & 1] : bb[PB & 1];
      const float bc = base[2 * (r & 1)], bs = base[2 * (r & 1) + 1];
      const float c = bc * ci[PB][r] - bs * si[PB][r], sn = bs * ci[PB][r] + bc * si[PB][r];
      kop[r] = from_f32<sc_t>(lo[r] * c - hi[r] * sn);
      kop[4 + r] = from_f32<sc_t>(hi[r] * c + lo[r] * sn);
    }
    return Elem<sc_t>::mfma16(kop, qop[PB], s);   // lane (head n16, g4): tokens 4 g4 + r
  };
  auto store = [&](int i, f32x4 s) {
    const int t = tok0 + i * STEP + 4 * g4;
    if (n16 >= G || t >= end) return;
    const int64_t o = ((int64_t)b * p.hq + h0 + n16) * p.kv_len + t;
    s *= p.sm_scale;
    if (vec_out && t + 4 <= end) {
      if (p.scores_dtype == XKV_F32) *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.scores) + o) = s;
      else *reinterpret_cast<vec4*>(reinterpret_cast<T*>(p.scores) + o) = vec4{from_f32<T>(s[0]), from_f32<T>(s[1]), from_f32<T>(s[2]), from_f32<T>(s[3])};
      return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (t + r < end) {
        if (p.scores_dtype == XKV_F32) reinterpret_cast<float*>(p.scores)[o + r] = s[r];
        else reinterpret_cast<T*>(p.scores)[o + r] = from_f32<T>(s[r]);
      }
  };
  // Deal the block's matrix instructions out among the rotation of the block before: left alone they come in one burst, and
  // a wave that issues in order then has both pipes wait for each other.
  auto interleave = [&]() {
    constexpr int VALU = (48 + 2 * NKS - 1) / (2 * NKS);
#pragma unroll
    for (int m = 0; m < 2 * NKS; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto step = [&](int i, auto buf_c) {   // tile i of this wave
    constexpr int B = decltype(buf_c)::value;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int cbk = 0; cbk < 8; ++cbk) asm volatile("" : "+a"(breg[ks][cbk]));
    load(i + NBUF - 1, IC<(B + NBUF - 1) % NBUF>());   // into the buffer tile i - 1 has left
    const float* bl = base_lds[wave][B & 1];
    *reinterpret_cast<float2*>(&base_lds[wave][B & 1][2 * lane]) = make_float2(cb, sb);
    {
      const float c = cb * c64 - sb * s64, s = sb * c64 + cb * s64;
      cb = c;
      sb = s;
    }
    // the row is written and read by this wave alone, whose LDS operations are carried out in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    auto read_base = [&](int pb) {
      const float* src = bl + (16 * pb + 4 * g4) * 2;
      ba[pb & 1] = *reinterpret_cast<const f32x4*>(src);
      bb[pb & 1] = *reinterpret_cast<const f32x4*>(src + 4);
    };
    read_base(0);
    rebuild(buf_c, IC<0>());
    s_prev = rotate_dot(IC<3>(), k[1][0], k[1][1], s_cur);   // the last block of tile i - 1
    interleave();
    read_base(1);
    rebuild(buf_c, IC<1>());
    s_cur = rotate_dot(IC<0>(), k[0][0], k[0][1], f32x4{0.f, 0.f, 0.f, 0.f});
    interleave();
    if (i > 0) store(i - 1, s_prev);
    read_base(2);
    rebuild(buf_c, IC<2>());
    s_cur = rotate_dot(IC<1>(), k[1][0], k[1][1], s_cur);
    interleave();
    read_base(3);
    rebuild(buf_c, IC<3>());
    s_cur = rotate_dot(IC<2>(), k[0][0], k[0][1], s_cur);
    interleave();
  };
  for (int i = 0; i < n; i += NBUF) {
    if (i % SEED == 0) sincosf((float)(p.pos_offset + start + (int64_t)i * STEP) * inv, &sb, &cb);
    step(i, IC<0>());
    if (i + 1 < n) step(i + 1, IC<1>());
    if (i + 2 < n) step(i + 2, IC<2>());
    if (i + 3 < n) step(i + 3, IC<3>());
  }
  store(n - 1, rotate_dot(IC<3>(), k[1][0], k[1][1], s_cur));
}

template <typename T>
int launch(const FastParams& p, const FactorOperand& kB, int batch, int rank, hipStream_t st) {
  const int vec_out = p.kv_len % 4 == 0 && (reinterpret_cast<uintptr_t>(p.scores) & 15) == 0;
  const dim3 grid(xcd_grid(batch * p.hkv * p.max_splits, p.hkv)), block(256);
  switch (rank / 32) {
#define XKV_SCORES_RANK(N) case N: recon_scores_kernel<T, N><<<grid, block, 0, st>>>(p, kB, vec_out); break;
    XKV_SCORES_RANK(1) XKV_SCORES_RANK(2) XKV_SCORES_RANK(3) XKV_SCORES_RANK(4) XKV_SCORES_RANK(5) XKV_SCORES_RANK(6)
#undef XKV_SCORES_RANK
    default: return XKV_EUNSUPPORTED;
  }
  return launch_status();
}

}  // namespace

int launch_recon_scores(const FastParams& p, const void* kB, int64_t sBb, int64_t sBh, int64_t sBr, int batch, int dtype, int rank,
                        hipStream_t st) {
  const FactorOperand f{kB, sBb, sBh, sBr};
  return dtype == XKV_BF16 ? launch<__bf16>(p, f, batch, rank, st) : launch<_Float16>(p, f, batch, rank, st);
}

}  // namespace xkv
