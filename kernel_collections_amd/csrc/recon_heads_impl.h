// Several kv heads per workgroup: fused reconstruct + RoPE + softmax + P.A stage 1 (rank RK, head_dim 128, the token basis shared by K and V), or the
// scaled scores alone.
//
// Four wavefronts, one per SIMD, each with all 512 registers of its lanes; accumulation registers hold the factors of the NH kv heads, 16 of the 64 rotate-half
// pairs (both halves of each) per wave and head.  A tile of 32 tokens is read once for all of them: the token rows' way from the L2 into the LDS, the operand
// reads and the transposed reads of P.A are shared by NH heads.  These are what the chip is short of: with one head per workgroup (recon_spec_impl.h) it runs at its
// power limit, and every byte moved takes the clock down.
//
// A wave does everything itself, dealt out among the NK * NH matrix instructions v_mfma_f32_32x32x16 of a period, so that every one of them has a few
// others in its shadow (a wave alone on its SIMD hides four or five vector instructions behind each, and pays 5 cycles for each beyond).  In period pp:
//   the k-steps of tile pp, operands read AHEAD k-steps before their use
//   rotation and q-dot of tile pp - 1 (whole keys, no partial sums to add), scores over the wave's 16 pairs into the LDS
//   transposed reads of tile pp - 1
//   ---- the barrier, the only one: scores and q^ written, tile pp + 1 landed, tile pp - 1 read
//   softmax and P.A of tile pp - 1: every wave computes P of all heads and its RK / 4 latent features
// The loads of a tile go straight to the LDS, a row at a time, spread evenly over the period between two barriers (in a burst they keep the LDS from the
// operand reads), into the slot of the tile that the first of the two barriers has done with: they have a period to two to arrive.  The next tile's
// operands are read behind the barrier that has waited for it (NEXT).
//
// 16 x 32768 tokens, 32 heads on 8 kv heads, several heads / one a workgroup: rank 512 446 / 528 us (438 / 506 at a higher clock: 1.30 PFLOP/s), 384 360 / 416, 256, four heads, 243; 2755 - 2785 clocks a
// period at rank 512 where the matrix instructions take 2240, at 1.57 - 1.62 GHz under the power limit (matrix instructions alone: 1.8).  A call starts with 16000 - 20000 clocks in front of the first period:
// 6000 until the first load of a cold device returns, then 256 KB of factors at the rate at which all CUs together read the L2 (33 bytes a clock each).
#pragma once
#include "recon_fast_impl.h"
#include <utility>

namespace xkv {
namespace heads {
using namespace fast;

typedef short s16x4h __attribute__((ext_vector_type(4)));
typedef short s16x8h __attribute__((ext_vector_type(8)));

constexpr int RING = 4;              // tiles in the LDS: the one in use, the one before it, the next one, the one on its way

// Places in a period of M matrix instructions
template <int RK, int NH, bool SCORES, int TPL> struct HeadsShape {
  static constexpr int FROW = RK * 2 + 16;     // LDS bytes per tile row
  static constexpr int FTILE = FT * FROW;
  static constexpr int NK = RK / 16, M = NK * NH;
  static constexpr int NMB = RK / 64;          // 16-feature blocks of the RK / 4 latent features a wave owns in P.A
  static constexpr int AHEAD = 10 / NH;        // k-steps between the read of an operand and its use
  static constexpr int SP_FLOATS = 4 * NH * 8 * FSP_ROW;   // one buffer of partial scores: [wave 4][kv NH][head 8][FSP_ROW]
  // rotation: QU instructions per quarter (four pairs a lane) of a head
  static constexpr bool FP32 = SCORES || RK == 256;   // rotation
  static constexpr int QU = FP32 ? 20 : 12, NU = QU * 2 * NH;
  static constexpr int SU = TPL / 4 * 7 + 2;   // steps of the softmax
  static constexpr int PA = (NMB + 1) / 2;     // places of P.A at the end
  static constexpr int ROT0 = NH + 3;
  static constexpr int NEXT = (NK - AHEAD) * NH;   // the next tile's operands are read from here on
  static constexpr int BAR = SCORES ? NEXT : M - PA - SU - 5 - (M >= 64 && TPL == 4 ? 2 : 0);
  static constexpr int ROT1 = BAR - 4;         // the last quarter's q-dot and its scores follow
  static constexpr int upto(int m) { return m <= ROT0 ? 0 : m >= ROT1 ? NU : (m - ROT0) * NU / (ROT1 - ROT0); }   // instructions in front of place m
  static constexpr int done(int q) { int m = 0; while (upto(m) < (q + 1) * QU) ++m; return m; }                     // quarter q is in front of this place
  static constexpr int S0 = BAR + 5;           // the softmax, its operands read from BAR + 1 on
  static constexpr int TR0 = BAR - 2 - 2 * NMB > 0 ? BAR - 2 - 2 * NMB : 0, TRN = BAR - 2 - TR0;   // transposed reads
  static constexpr size_t SHM = (size_t)RING * FTILE + 2 * SP_FLOATS * 4 + 2 * NH * 8 * 128 * 2 + 128 * 2 + NH * 8 * 4;
};

// GP: head slots of a kv head (4 or 8).  SCORES: write the scaled scores only.
template <typename T, bool SCORES, int RK, int GP, int NH>
__global__ __launch_bounds__(256, 1) void recon_heads_kernel(const FastParams p, const FactorOperand kB) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int GC = NH * GP;                  // head slots of the workgroup
  constexpr int TPL = GC / 2;                  // tokens per lane of the softmax
  typedef HeadsShape<RK, NH, SCORES, TPL> S;
  constexpr int FROW = S::FROW, FTILE = S::FTILE, NK = S::NK, M = S::M, NMB = S::NMB, SP_FLOATS = S::SP_FLOATS, AHEAD = S::AHEAD, BAR = S::BAR, QU = S::QU;
  constexpr bool FP32 = S::FP32;
  static_assert(GC <= 16 && GC >= 8 && (S::ROT1 - S::ROT0) > 0 && S::done(2 * NH - 1) + 2 < BAR && BAR <= S::NEXT, "places of a period");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n32 = lane & 31, g2 = lane >> 5;
  const int n16 = lane & 15, g4 = lane >> 4;

  const int ngroups = p.hkv / NH;
  const int wg = xcd_cluster_remap(blockIdx.x, ngroups);   // the heads of one (sequence, split) stream the same rows: one L2
  if (wg >= p.total_wg) return;
  const int kh = NH * (wg % ngroups);
  const int split = (wg / ngroups) % p.max_splits;
  const int b = wg / (ngroups * p.max_splits);
  const int L = p.kv_lens ? p.kv_lens[b] : p.kv_len;
  int start, end;
  split_bounds(L, asked_splits(p.num_splits, b, p.max_splits, 0), split, start, end);
  if (end <= start) return;
  const int G = p.hq / p.hkv, h0 = kh * G;
  const int ntiles = (end - start + FT - 1) / FT;

  unsigned char* ring = smem;
  float* s_part = reinterpret_cast<float*>(smem + RING * FTILE);           // [2][4 waves][NH][8 heads][FSP_ROW]
  sc_t* qhat = reinterpret_cast<sc_t*>(s_part + 2 * SP_FLOATS);            // [2][NH][8 heads][128]
  constexpr int QPART = NH * 8 * 128;
  sc_t* qzero = qhat + 2 * QPART;                                      // [128] zeros: the q-dot operand of masked lanes
  float* unscale = reinterpret_cast<float*>(qzero + 128);                  // [NH][8]
  const unsigned ring_lds = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)ring;

  // ---- what is read of queries and frequencies: in front of the loads that take longer
  constexpr int QH = GC / 4;
  T qraw[QH][2];
#pragma unroll
  for (int i = 0; i < QH; ++i) {
    const int s = wave + 4 * i, kv = s / GP, g = s % GP;
    const T* qrow = reinterpret_cast<const T*>(p.q) + ((int64_t)b * p.hq + h0 + kv * G + (g < G ? g : 0)) * 128 + lane;
    qraw[i][0] = qrow[0];
    qraw[i][1] = qrow[64];
  }
  const float qinv = p.inv_freq[lane];
  float freq[8];           // of this lane's pairs 16 wave + 8 (r / 4) + 4 g2 + r % 4
#pragma unroll
  for (int r = 0; r < 8; ++r) freq[r] = p.inv_freq[16 * wave + 8 * (r >> 2) + 4 * g2 + (r & 3)];
  XKV_FENCE();
  // ---- the factors, CH ranks of a head at a time through the LDS behind the first tiles (in memory a rank is a row, the operand wants
  // consecutive ranks in a lane), into accumulation registers: lane (feature 64 (n32 / 16) + 16 wave + n16, g2) holds 8 consecutive ranks
  vec8 breg[NH][NK];
  constexpr int CH = 64, CLD = 128 + 8, NCH = NH * RK / CH, DEEP = 8;   // DEEP: chunks on the way
  static_assert(FTILE + 2 * SP_FLOATS * 4 >= 2 * CH * CLD * 2, "room for two chunks");
  const T* Bh = reinterpret_cast<const T*>(kB.p) + b * kB.sb + kh * kB.sh + (int64_t)(tid >> 4) * kB.sr + (tid & 15) * 8;
  T* stage = reinterpret_cast<T*>(ring + (RING - 1) * FTILE);
  vec8 rows[DEEP][4];
  auto fetch = [&](auto c_c) {
    constexpr int C = decltype(c_c)::value;
    if constexpr (C < NCH) {
#pragma unroll
      for (int i = 0; i < 4; ++i) rows[C % DEEP][i] = ld16<vec8>(Bh + (C / (RK / CH)) * kB.sh + (int64_t)(C % (RK / CH) * CH + 16 * i) * kB.sr);
    }
  };
  static_for<DEEP>(fetch);
  XKV_FENCE();
  // ---- tile loads: rows 8 wave .. + 7 of a tile are this wave's.  Rows past the split's end are out of the resource's range and leave zeros
  const int row_bytes = (int)p.sAl * 2;
  const unsigned char* arow = reinterpret_cast<const unsigned char*>(p.kA) + (b * p.sAb + (int64_t)(start + 8 * wave) * p.sAl) * 2;
  int aleft = end - start - 8 * wave;    // rows of the split from arow on
  const unsigned row_lds = ring_lds + wave * 8 * FROW, lane16 = lane * 16;
  u32x4 ares;
  auto next_tile = [&]() {
    const int have = aleft < 8 ? aleft : 8;
    const uint64_t at = reinterpret_cast<uint64_t>(arow);
    ares = u32x4{(unsigned)__builtin_amdgcn_readfirstlane((unsigned)at), (unsigned)__builtin_amdgcn_readfirstlane((unsigned)(at >> 32) & 0xffff),
                 (unsigned)__builtin_amdgcn_readfirstlane(have > 0 ? (have - 1) * row_bytes + RK * 2 : 0), 0x00020000u};
    arow += (int64_t)FT * row_bytes;
    aleft -= FT;
  };
  auto load_row = [&](auto slot_c, auto r_c) {
    constexpr int R = decltype(r_c)::value;
    row_to_lds<RK, decltype(slot_c)::value * FTILE + R * FROW>(ares, lane16, R * row_bytes, row_lds);
  };
  static_for<RING - 1>([&](auto t_c) {
    next_tile();
    static_for<8>([&](auto r_c) { load_row(t_c, r_c); });
  });
  if (tid < 128) qzero[tid] = from_f32<sc_t>(0.f);
  // ---- in-tile rotation of this wave's 8 pairs per lane (token n32, g2): pair 16 wave + 8 (r / 4) + 4 g2 + r % 4, r = 0 .. 7.  Two tables: the
  // query-side base is that of an EVEN tile and serves the odd tile after it too, whose offsets are 32 .. 63.
  float ct[2][8], st[2][8];
  h2 ch[2][4], sh[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 8; ++r)
      __sincosf((float)(n32 + 32 * h) * freq[r], &st[h][r], &ct[h][r]);
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      ch[h][k] = h2{(_Float16)ct[h][2 * k], (_Float16)ct[h][2 * k + 1]};
      sh[h][k] = h2{(_Float16)st[h][2 * k], (_Float16)st[h][2 * k + 1]};
    }
  // ---- query-side base rotation: lane = pair, head slots wave, wave + 4, ...
  float q0[QH], q1[QH];
#pragma unroll
  for (int i = 0; i < QH; ++i) {
    const int s = wave + 4 * i, kv = s / GP, g = s % GP;
    q0[i] = g < G ? to_f32(qraw[i][0]) : 0.f;
    q1[i] = g < G ? to_f32(qraw[i][1]) : 0.f;
    // Multiplied by the power of two that brings the head's largest feature to 2^14 .. 2^15, and the scores by the inverse: fp16 then holds every
    // rotated pair, and the parts of small queries are no subnormals there.  A feature that is no finite number leaves the others as they are.
    const int bits = __builtin_bit_cast(int, row_reduce<true, 16>(fmaxf(fabsf(q0[i]), fabsf(q1[i]))));
    const int top = max(max(__builtin_amdgcn_readlane(bits, 0), __builtin_amdgcn_readlane(bits, 16)),
                        max(__builtin_amdgcn_readlane(bits, 32), __builtin_amdgcn_readlane(bits, 48)));
    const int up = max(-1, min(14 + 127 - (top >> 23), 100));
    const float f = __builtin_bit_cast(float, (127 + up) << 23);
    q0[i] *= f;
    q1[i] *= f;
    if (lane == 0) unscale[kv * 8 + g] = __builtin_bit_cast(float, (127 - up) << 23);
  }
  // q^ is kept in q-dot operand order: pair j = 32 dq' + 8 o + 4 g' + e sits at [o][dq'][g'][e] (partner at e + 4)
  const int qpos = ((((lane >> 3) & 3) * 2 + (lane >> 5)) * 2 + ((lane >> 2) & 1)) * 8 + (lane & 3);
  float qc64, qs64, qcb, qsb;   // (qcb, qsb): base rotation of the tiles whose q^ is written next
  sincosf((float)(2 * FT) * qinv, &qs64, &qc64);
  auto seed_qhat = [&](int t) { sincosf((float)(p.pos_offset + start + (int64_t)t * FT) * qinv, &qsb, &qcb); };
  // q^ for the even tile t and the odd one after it = R(-base(t)) q, into buffer (t / 2) & 1
  auto write_qhat = [&](int t, auto i_c) {
    constexpr int I = decltype(i_c)::value;
    const int s = wave + 4 * I;
    sc_t* d = qhat + ((t >> 1) & 1) * QPART + qpos + ((s / GP) * 8 + s % GP) * 128;
    const float r0 = q0[I] * qcb + q1[I] * qsb, r1 = q1[I] * qcb - q0[I] * qsb;
    d[0] = from_f32<sc_t>(r0);
    d[4] = from_f32<sc_t>(r1);
    if constexpr (I == QH - 1) {
      const float cc = qcb * qc64 - qsb * qs64, ss = qsb * qc64 + qcb * qs64;
      qcb = cc; qsb = ss;
    }
  };
  seed_qhat(0);
  static_for<QH>([&](auto i_c) { write_qhat(0, i_c); });
  // ---- the factors, from registers through the LDS into accumulation registers
  static_for<NCH>([&](auto c_c) {
    constexpr int C = decltype(c_c)::value, KV = C / (RK / CH), KS0 = C % (RK / CH) * (CH / 16);
    T* buf = stage + (C % 2) * CH * CLD;
#pragma unroll
    for (int i = 0; i < 4; ++i) st16(buf + ((tid >> 4) + 16 * i) * CLD + (tid & 15) * 8, rows[C % DEEP][i]);
    fetch(IC<C + DEEP>());
    __syncthreads();   // whoever is here has read the chunk before, whose place the next one takes
#pragma unroll
    for (int ks = 0; ks < CH / 16; ++ks) {
      const T* src = buf + (16 * ks + 8 * g2 + (n16 >> 2)) * CLD + 64 * (n32 >> 4) + 16 * wave + 4 * (n16 & 3);
      const s16x4h lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4h*)src);
      const s16x4h hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4h*)(src + 4 * CLD));
      breg[KV][KS0 + ks] = __builtin_bit_cast(vec8, (s16x8h)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      asm volatile("" : "+a"(breg[KV][KS0 + ks]));
    }
  });
  __syncthreads();
  // q-dot B operand: lanes whose token half (lane bit 4) matches their column's (lane bit 3) read q^ of head lane % 8 (absent heads: the
  // last one; their columns are not used), the others read zeros
  const bool q_live = ((lane >> 4) & 1) == ((lane >> 3) & 1);
  const sc_t* qsrc = q_live ? qhat + ((lane & 7) < G ? (lane & 7) : G - 1) * 128 + ((wave & 1) * 4 + (wave >> 1)) * 16 + g2 * 8 : qzero;
  const int qpar = q_live ? QPART : 0, qkv = q_live ? 8 * 128 : 0;
  float* const sdst = s_part + (wave * NH * 8 + (n16 & 7)) * FSP_ROW + 16 * (n16 >> 3) + 4 * g4;

  // ---- softmax role: lane (n16, g4) holds head slot n16 % GC, tokens 8 g4 + TPL (n16 / GC) ..
  const int sm_slot = n16 & (GC - 1), sm_g = sm_slot % GP;
  const int sm_tok = 8 * g4 + TPL * (n16 / GC);
  const float* const ssrc = s_part + ((sm_slot / GP) * 8 + (sm_g < G ? sm_g : G - 1)) * FSP_ROW + sm_tok;
  float m_ref = NEG_INF, l_run = 0.f;   // reference maximum of the lane's head (base-2 domain); this lane's share of its row sum
  // Rank 256: the running maximum itself, whose weight of 1 is exact in 16 bits, as in the pass over given scores that long calls had before.  65536 tokens, 32 heads on 8 kv heads:
  // 50.4 us a call, 49.4 with a lazy reference, 58.8 as two passes; error of bf16 against float64 3.2e-4, 3.6e-4, 3.0e-4 over even weights, 1.1e-3, 1.7e-3, 1.1e-3 over peaked ones
  constexpr float LAZY = RK == 256 ? 0.f : lazy_rescale<T>();
  const float scale2 = p.sm_scale * unscale[(sm_slot / GP) * 8 + (sm_g < G ? sm_g : G - 1)] * 1.44269504088896f, lazy2 = LAZY * 1.44269504088896f;
  f32x4 acc[NMB];
#pragma unroll
  for (int mb = 0; mb < NMB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Transposed reads: a 16-lane group reads a block of 4 rows x 16 columns.  Rows 2 j (first read) and 2 j + 1 (second read) of the group's 8 tokens: with
  // the 16-byte row padding, rows two apart do not overlap in the banks.  Element e of the lane's 8 contraction values is token 8 g4 + 2 e (e < 4) or
  // 8 g4 + 2 (e - 4) + 1.
  const unsigned char* trsrc = ring + (8 * g4 + 2 * (n16 >> 2)) * FROW + (wave * (RK / 4) + 4 * (n16 & 3)) * 2;

  f32x16 k[2][NH];         // [parity of the tile][kv]: registers 0 .. 7 the low features of the lane's pairs, 8 .. 15 their partners
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int kv = 0; kv < NH; ++kv)
#pragma unroll
      for (int r = 0; r < 16; ++r) k[s][kv][r] = 0.f;
  const unsigned char* fr0 = ring + n32 * FROW + 8 * g2 * 2;
  // period 0 multiplies a tile that does not exist, in the last slot, by zeros
  if constexpr (!SCORES)
    for (int i = tid * 16; i < FTILE; i += 256 * 16) *reinterpret_cast<u32x4*>(ring + (RING - 1) * FTILE + i) = u32x4{0, 0, 0, 0};
  wait_vmcnt<0>();
  __syncthreads();

  vec8 at[NK];             // operands on the way or waiting
  auto read_operand = [&](auto slot_c, auto ks_c) {
    constexpr int KS = decltype(ks_c)::value;
    at[KS] = ld16<vec8>(fr0 + decltype(slot_c)::value * FTILE + KS * 32);
  };
  static_for<AHEAD>([&](auto ks_c) { read_operand(IC<0>(), ks_c); });

  auto here = [](auto& v) { asm volatile("" : "+v"(v)); };   // computed at this place: without it the compiler moves chains together
  s16x4h tr[2 * NMB];      // tile pp - 1 transposed
  auto period = [&](int pp, auto u_c) {
    constexpr int u = decltype(u_c)::value, PAR = u & 1;
#pragma unroll
    for (int kv = 0; kv < NH; ++kv)
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) asm volatile("" : "+a"(breg[kv][ks]));
    const int t1 = pp - 1;
    const bool live = pp > 0;
    // rotation of tile pp - 1, four pairs of a head at a time, in three stages that depend on the stage before alone.  Scores, and rank 256, whose long calls
    // took their scores apart before: in fp32, rounded once.  Else in packed fp16 (its error is that of the keys' rounding once more).  Rank 256, 65536 tokens, 32 heads on 8
    // kv heads: 49.4 us a call in fp32, 47.7 in fp16 
    float tl[4], th[4], kl[4], kr[4];
    h2 lo2[2], hi2[2], pl[2], ph[2], kw[4];
    auto rotate = [&](auto u2_c) {
      constexpr int KV = decltype(u2_c)::value / (2 * QU), O = decltype(u2_c)::value / QU % 2, U = decltype(u2_c)::value % QU;
      const f32x16& j = k[PAR ^ 1][KV];
      if constexpr (FP32) {
        constexpr int STAGE = U / 8, R = STAGE < 2 ? U % 8 / 2 : U - 16;
        const float lo = j[4 * O + R], hi = j[8 + 4 * O + R], cc = ct[PAR ^ 1][4 * O + R], ss = st[PAR ^ 1][4 * O + R];
        if constexpr (STAGE == 0) {
          if constexpr (U % 2 == 0) { tl[R] = hi * ss; here(tl[R]); }
          else { th[R] = lo * ss; here(th[R]); }
        } else if constexpr (STAGE == 1) {
          if constexpr (U % 2 == 0) { kl[R] = __builtin_fmaf(lo, cc, -tl[R]); here(kl[R]); }
          else { kr[R] = __builtin_fmaf(hi, cc, th[R]); here(kr[R]); }
        } else {
          if constexpr (R < 2) kw[R] = h2{(_Float16)kl[2 * R], (_Float16)kl[2 * R + 1]};
          else kw[R] = h2{(_Float16)kr[2 * R - 4], (_Float16)kr[2 * R - 3]};
          here(kw[R]);
        }
      } else {
        constexpr int STAGE = U / 4, E = U % 4 / 2;
        const h2 cc = ch[PAR ^ 1][2 * O + E], ss = sh[PAR ^ 1][2 * O + E];
        if constexpr (STAGE == 0) {
          if constexpr (U % 2 == 0) { lo2[E] = h2{(_Float16)j[4 * O + 2 * E], (_Float16)j[4 * O + 2 * E + 1]}; here(lo2[E]); }
          else { hi2[E] = h2{(_Float16)j[8 + 4 * O + 2 * E], (_Float16)j[8 + 4 * O + 2 * E + 1]}; here(hi2[E]); }
        } else if constexpr (STAGE == 1) {
          if constexpr (U % 2 == 0) { pl[E] = hi2[E] * ss; here(pl[E]); }
          else { ph[E] = lo2[E] * ss; here(ph[E]); }
        } else {
          if constexpr (U % 2 == 0) { kw[E] = lo2[E] * cc - pl[E]; here(kw[E]); }
          else { kw[2 + E] = hi2[E] * cc + ph[E]; here(kw[2 + E]); }
        }
      }
    };
    // q-dot.  As the A operand of v_mfma_f32_16x16x32, lane (n32, g2) is row n32 % 16 and k-group (n32 / 16) + 2 g2; the B operand
    // keeps the token halves apart (column c' holds q^ of head c' % 8 in the k-groups of token half c' / 8, zeros elsewhere).
    // Result: lane (c', g4), register r = score of token 16 (c' / 8) + 4 g4 + r for head c' % 8.
    sc_vec8 qop[2];
    f32x4 sacc[2];
    auto read_q = [&](auto q_c) {
      constexpr int KV = decltype(q_c)::value / 2, O = decltype(q_c)::value % 2;
      qop[O] = ld16<sc_vec8>(qsrc + (((pp - 1) >> 1) & 1) * qpar + KV * qkv + O * 32);
    };
    auto dot = [&](auto q_c) {
      constexpr int KV = decltype(q_c)::value / 2, O = decltype(q_c)::value % 2;
      const sc_vec8 kop = {kw[0][0], kw[0][1], kw[1][0], kw[1][1], kw[2][0], kw[2][1], kw[3][0], kw[3][1]};
      sacc[KV & 1] = Elem<sc_t>::mfma16(kop, qop[O], O == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sacc[KV & 1]);
    };
    // softmax of tile pp - 1
    typedef float fv __attribute__((ext_vector_type(4)));
    constexpr int NV = TPL / 4;
    fv part[4][NV], sa[NV], sb[NV];
    float s[TPL], e[TPL];
    u32x4 pbu;
    auto softmax = [&](auto i_c) {
      constexpr int I = decltype(i_c)::value;
      if constexpr (I < NV) { sa[I] = part[0][I] + part[1][I]; here(sa[I]); }
      else if constexpr (I < 2 * NV) { sb[I - NV] = part[2][I - NV] + part[3][I - NV]; here(sb[I - NV]); }
      else if constexpr (I < 3 * NV) { sa[I - 2 * NV] += sb[I - 2 * NV]; here(sa[I - 2 * NV]); }
      else if constexpr (I < 4 * NV) {
#pragma unroll
        for (int x = 0; x < 4; ++x) { s[4 * (I - 3 * NV) + x] = sa[I - 3 * NV][x] * scale2; here(s[4 * (I - 3 * NV) + x]); }
      } else if constexpr (I == 4 * NV) {
        const int tok = start + t1 * FT + sm_tok;
        if (start + t1 * FT + FT > end || !live) {   // the split's last tile, and the one before its first
#pragma unroll
          for (int x = 0; x < TPL; ++x) if (tok + x >= end || !live) s[x] = NEG_INF;
        }
        float mxl = s[0];
#pragma unroll
        for (int x = 1; x < TPL; ++x) mxl = fmaxf(mxl, s[x]);
        // the reference maximum only moves when the tile maximum exceeds it by the lazy bound; the cross-lane reduction that
        // finds the maximum runs only then.  Every wave sees the same scores, so all four keep the same reference.
        if (__builtin_amdgcn_ballot_w64(mxl > m_ref + lazy2)) {
          float mx = mxl;
#pragma unroll
          for (int m = GC; m < 64; m <<= 1) mx = fmaxf(mx, __shfl_xor(mx, m));
          const float m_new = mx > m_ref + lazy2 ? mx : m_ref;
          const float alpha = __builtin_amdgcn_exp2f(m_ref - m_new);
          m_ref = m_new;
          l_run *= alpha;
#pragma unroll
          for (int mb = 0; mb < NMB; ++mb) acc[mb] *= alpha;   // column n16 of the accumulators is this lane's head
        }
      } else if constexpr (I <= 5 * NV) {
#pragma unroll
        for (int x = 0; x < 4; ++x) { float& y = s[4 * (I - 4 * NV - 1) + x]; y -= m_ref; here(y); }
      } else if constexpr (I <= 6 * NV) {
#pragma unroll
        for (int x = 0; x < 4; ++x) { float& y = e[4 * (I - 5 * NV - 1) + x]; y = __builtin_amdgcn_exp2f(s[4 * (I - 5 * NV - 1) + x]); here(y); }
      } else if constexpr (I <= 7 * NV) {
        if constexpr (I == 6 * NV + 1) {
          // P of the tile that does not exist: its scores are no numbers, minus infinity less minus infinity
          if (!live) {
#pragma unroll
            for (int x = 0; x < TPL; ++x) e[x] = 0.f;
          }
        }
        const int x = 4 * (I - 6 * NV - 1);
        l_run += (e[x] + e[x + 1]) + (e[x + 2] + e[x + 3]);
      } else {
        // P as the B operand of v_mfma_f32_16x16x32: lane (column n16 = head slot, g4) holds its head's tokens 8 g4 .. + 8 in the order
        // of the transposed reads (even tokens, then odd ones)
        if constexpr (GC == 8) {
          const unsigned ev = pack_pair<T>(e[0], e[2]), od = pack_pair<T>(e[1], e[3]);
          pbu = u32x4{ev, dpp_u32<0x108>(ev), od, dpp_u32<0x108>(od)};
        } else {
          pbu = u32x4{pack_pair<T>(e[0], e[2]), pack_pair<T>(e[TPL - 4], e[TPL - 2]), pack_pair<T>(e[1], e[3]), pack_pair<T>(e[TPL - 3], e[TPL - 1])};
        }
        here(pbu);
      }
    };
    // scores out: lane -> (head slot 2 wave + 8 i + lane / 32, token lane % 32)
    float so[GC / 8][4];
    static_for<M>([&](auto m_c) {
      constexpr int m = decltype(m_c)::value, v = m / NH, i = m % NH;
      if constexpr (m == BAR) {
        wait_vmcnt<8>();   // the loads since the last barrier are those of tile pp + 2
        __syncthreads();
        next_tile();
      }
      if constexpr (v == 0) {
        const f32x16 z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        k[PAR][i] = Elem<T>::mfma32(breg[i][0], at[0], z);
      } else {
        k[PAR][i] = Elem<T>::mfma32(breg[i][v], at[v], k[PAR][i]);
      }
      if constexpr (i == 0) read_operand(IC<v + AHEAD < NK ? u : (u + 1) % RING>(), IC<(v + AHEAD) % NK>());
      // ---- q-dots, rotation
      static_for<2 * NH>([&](auto q_c) {
        constexpr int q = decltype(q_c)::value, D = S::done(q);
        if constexpr (m == D) dot(q_c);
        if constexpr (q % 2 == 1 && m == D + 2) *reinterpret_cast<f32x4*>(sdst + (PAR ^ 1) * SP_FLOATS + (q / 2) * 8 * FSP_ROW) = sacc[(q / 2) & 1];
        constexpr int RD = q < 2 ? 1 + q : S::done(q - 2) + 1;   // its operand, as soon as that of the quarter before the last is used
        if constexpr (m == RD) read_q(q_c);
      });
      static_for<S::upto(m + 1) - S::upto(m)>([&](auto j_c) { rotate(IC<S::upto(m) + decltype(j_c)::value>()); });
      // ---- tile loads: the first rows of tile pp + 3 behind the barrier, the others, of tile pp + 2, in front of the next one
      constexpr int LSTEP = M / 8, L0 = LSTEP / 2, LB = (BAR + LSTEP - 1 - L0) / LSTEP;   // LB: rows in front of the barrier
      if constexpr (m % LSTEP == L0) {
        if constexpr (m >= BAR) load_row(IC<(u + 3) % RING>(), IC<m / LSTEP - LB>());
        else load_row(IC<(u + 2) % RING>(), IC<m / LSTEP + 8 - LB>());
      }
      if constexpr (!SCORES) {
        if constexpr (m >= S::TR0 && m < S::TR0 + S::TRN) {
          static_for<2 * NMB>([&](auto r_c) {
            constexpr int r = decltype(r_c)::value;
            if constexpr (S::TR0 + r * S::TRN / (2 * NMB) == m)
              tr[r] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4h*)(trsrc + ((u + 3) % RING) * FTILE + (r / 2) * 32 + (r % 2) * FROW));
          });
        }
        if constexpr (m >= BAR && m < BAR + 4) {
#pragma unroll
          for (int x = 0; x < NV; ++x) part[m - BAR][x] = *reinterpret_cast<const fv*>(ssrc + (PAR ^ 1) * SP_FLOATS + (m - BAR) * NH * 8 * FSP_ROW + 4 * x);
        }
        if constexpr (m >= S::S0 && m < S::S0 + S::SU) softmax(IC<m - S::S0>());
        constexpr int P0 = S::S0 + S::SU, PN = M - P0;
        if constexpr (m >= P0)
          static_for<NMB>([&](auto b_c) {
            constexpr int MB = decltype(b_c)::value;
            if constexpr (P0 + MB * PN / NMB == m)
              acc[MB] = Elem<T>::mfma16(__builtin_bit_cast(vec8, (s16x8h)__builtin_shufflevector(tr[2 * MB], tr[2 * MB + 1], 0, 1, 2, 3, 4, 5, 6, 7)),
                                        __builtin_bit_cast(vec8, pbu), acc[MB]);
          });
      } else {
        if constexpr (m == BAR) {
#pragma unroll
          for (int x = 0; x < GC / 8; ++x) {
            const int slot = 2 * wave + 8 * x + g2, g = slot % GP;
            const float* sp = s_part + (PAR ^ 1) * SP_FLOATS + ((slot / GP) * 8 + (g < G ? g : G - 1)) * FSP_ROW + n32;
#pragma unroll
            for (int w = 0; w < 4; ++w) so[x][w] = sp[w * NH * 8 * FSP_ROW];
          }
        }
        if constexpr (m == BAR + 3) {
#pragma unroll
          for (int x = 0; x < GC / 8; ++x) {
            const int slot = 2 * wave + 8 * x + g2, kv = slot / GP, g = slot % GP;
            const float y = ((so[x][0] + so[x][1]) + (so[x][2] + so[x][3])) * (p.sm_scale * unscale[kv * 8 + g]);
            const int tok = start + t1 * FT + n32;
            if (g < G && live && tok < end) {
              const int64_t o = ((int64_t)b * p.hq + h0 + kv * G + g) * p.kv_len + tok;
              if (p.scores_dtype == XKV_F32) reinterpret_cast<float*>(p.scores)[o] = y;
              else reinterpret_cast<T*>(p.scores)[o] = from_f32<T>(y);
            }
          }
        }
      }
      if constexpr (PAR == 0 && m >= 1 && m <= QH) { if (pp > 0) write_qhat(pp, IC<m - 1>()); }
      XKV_FENCE();
    });
  };
  for (int pb = 0;; pb += RING) {   // periods 0 .. ntiles
    if (pb > 0 && pb % 28 == 0) seed_qhat(pb);   // period pb writes q^ of tile pb next
    period(pb, IC<0>());
    if (pb + 1 > ntiles) break;
    period(pb + 1, IC<1>());
    if (pb + 2 > ntiles) break;
    period(pb + 2, IC<2>());
    if (pb + 3 > ntiles) break;
    period(pb + 3, IC<3>());
    if (pb + 4 > ntiles) break;
  }
  wait_vmcnt<0>();   // tiles past the end: none may arrive in a place that is another workgroup's by then
  if (SCORES) return;

  float l_head = l_run;
#pragma unroll
  for (int m = GC; m < 64; m <<= 1) l_head += __shfl_xor(l_head, m);
  // the lane's number once more, so that nothing lives through the loop for this
  int el = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  asm volatile("" : "+v"(el));
  const int e16 = el & 15, e4 = el >> 4, kv = (e16 & (GC - 1)) / GP, g = e16 % GP;
  if (e16 < GC && g < G) {
    const float inv = 1.f / l_head;
    const int64_t ph = ((int64_t)b * p.hq + h0 + kv * G + g) * p.max_splits + split;
    float* dst = p.partial + ph * RK + wave * (RK / 4) + 4 * e4;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) *reinterpret_cast<f32x4*>(dst + mb * 16) = acc[mb] * inv;
    if (wave == 0 && e4 == 0) p.lse[ph] = m_ref * 0.6931471805599453f + __logf(l_head);
  }
}

}  // namespace heads
}  // namespace xkv
