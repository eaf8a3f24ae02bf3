// Wave-specialised form of the fused reconstruct + RoPE + softmax + P.A stage 1 (rank RK = 512 / 384 / 256, head_dim 128,
// the token basis shared by K and V), one kv head per workgroup: 8 wavefronts, two per SIMD, with different jobs.
//
// Reconstruction waves (0..3): wave w keeps the 16 rotate-half pairs 16 w .. of B_h, both halves of each, over all ranks, stationary in
// RK / 4 accumulation registers, one v_mfma_f32_32x32x16 a k-step of the 32-token tile.  A lane then has whole pairs of one token, so the wave
// rotates them itself, in fp32 in the shadow of the next tile's matrix instructions, and takes their part of the q-dot: what it hands
// over is scores, 4 KB a tile.  It also sends the tile loads, evenly spread.  (Split 2 x 2 over rank and feature halves, each operand read served two matrix
// instructions, but 16 KB of partial keys went through the LDS and back, whose writes wait while load data arrives, and the consumers added and
// rotated them: 521 us for 16 x 32768 tokens, 8 kv heads, rank 512, against 506; 1 x 1000 22.3 / 21.4 a call, 4096 25.5 / 24.1, 30000 on one kv head 28.3 / 26.7,
// 130000 on three 75.5 / 72.3; rank 384, 2 x 50000 on three 51.7 / 46.8; rank 256, 64 heads on 8, 40000 47.3 / 40.2.  Then without a launch in front that packed the factor:
// 1 x 1000 19.9, 4096 22.1.)
// Consumer waves (4..7; consumer c owns RK / 4 latent features of P.A) do the rest, each step one workgroup barrier behind the one before it:
//   period p:  reconstruction   last k-steps of tile p-1, rotation + q-dot of tile p-1, first k-steps of tile p, loads of tile p+3 (ring of 4 slots)
//              consumers        softmax + P.A of tile p-2 (scores summed from the four waves' parts; the softmax is computed by
//                               every consumer for all heads, so P goes from registers straight into the MFMA operand),
//                               transposed reads of tile p for its P.A, kept in accumulation registers until period p+2 (2 sets of RK / 16),
//                               q^ for the next pair of tiles (even p)
// One barrier per period is the only synchronisation: everything a period reads was written at least one barrier earlier.  A tile is read from the LDS in
// one period only (reconstruction and transposed reads run in period p).
// What bounds it: the power limit.  A period of 1577 clocks against 1832 before took 0.97 of the time, the clock down from 1.8 to 1.57 GHz under the bytes that
// each kv head moves for itself; where several kv heads can share them, recon_heads_impl.h takes the call.
#pragma once
#include "recon_fast_impl.h"
#include "factor_rows.h"

namespace xkv {
namespace spec {
using namespace fast;

constexpr int SRING = 4;
template <int RK> struct SpecShape {
  static_assert(RK == 512 || RK == 384 || RK == 256, "rank");
  static constexpr int FROW = RK * 2 + 16;     // LDS bytes per tile row
  static constexpr int FTILE = FT * FROW;
  static constexpr int NK = RK / 16;           // k-steps of a tile, one matrix instruction of a reconstruction wave each
  static constexpr int NMB = RK / 64;          // 16-feature blocks of the RK / 4 latent features a consumer owns in P.A
  static constexpr int SP_FLOATS = 4 * 8 * FSP_ROW;   // one buffer of partial scores: [reconstruction wave 4][head 8][FSP_ROW]
  static constexpr int LATE = 4;               // k-steps of a tile that run after the barrier that ends its period
  static constexpr int EARLY = 1;              // operand reads are issued this many slots before the uniform one-per-slot rate
  static constexpr size_t SHM = (size_t)SRING * FTILE + 2 * SP_FLOATS * 4 + 2 * 8 * 128 * 2 + 128 * 2 + 8 * 4;
};

// The consumer's accumulation registers are managed by hand, by register number, in asm statements: a[0 .. RK/16) hold the P.A
// accumulators (block mb in a[4 mb .. 4 mb + 3]), a[RK/16 .. 3 RK/16) two sets of transposed tile reads (set s, block mb in
// a[RK/16 (1 + s) + 4 mb .. + 3]).  The compiler must not manage them: the reads are in flight for a period (a register copy
// it inserted would copy stale contents), and it picks one register class for all MFMA results of a kernel.  Its own code
// in the consumer branch uses no accumulation register (the build checks the consumer's ordinary registers do not spill).
// Nothing reads an accumulator sooner than a barrier after the MFMA that wrote it, so no wait states are needed there.
// The first MFMA of a tile follows the VALU instructions that formed pb; as asm it gets no hazard handling from the compiler,
// so the wait states a VALU result needs before an MFMA may read it are part of the statement.
template <typename T, int ACC, int A> __device__ __forceinline__ void pa_mfma_at(u32x4 pb) {
  if constexpr (std::is_same<T, __bf16>::value) {
    if constexpr (ACC == 0)
      asm volatile("s_nop 7\n\tv_mfma_f32_16x16x32_bf16 a[%1:%2], a[%3:%4], %0, a[%1:%2]" ::"v"(pb), "n"(ACC), "n"(ACC + 3), "n"(A), "n"(A + 3));
    else
      asm volatile("v_mfma_f32_16x16x32_bf16 a[%1:%2], a[%3:%4], %0, a[%1:%2]" ::"v"(pb), "n"(ACC), "n"(ACC + 3), "n"(A), "n"(A + 3));
  } else {
    if constexpr (ACC == 0)
      asm volatile("s_nop 7\n\tv_mfma_f32_16x16x32_f16 a[%1:%2], a[%3:%4], %0, a[%1:%2]" ::"v"(pb), "n"(ACC), "n"(ACC + 3), "n"(A), "n"(A + 3));
    else
      asm volatile("v_mfma_f32_16x16x32_f16 a[%1:%2], a[%3:%4], %0, a[%1:%2]" ::"v"(pb), "n"(ACC), "n"(ACC + 3), "n"(A), "n"(A + 3));
  }
}
template <int R, int OFF> __device__ __forceinline__ void tr_read_at(unsigned addr) {
  asm volatile("ds_read_b64_tr_b16 a[%1:%2], %0 offset:%3" ::"v"(addr), "n"(R), "n"(R + 1), "n"(OFF) : "memory");
}
template <int R> __device__ __forceinline__ void acc_set_at(float x) { asm volatile("v_accvgpr_write_b32 a%1, %0" ::"v"(x), "n"(R)); }
template <int R> __device__ __forceinline__ float acc_get_at() {
  float x;
  asm volatile("v_accvgpr_read_b32 %0, a%1" : "=v"(x) : "n"(R));
  return x;
}
// GP: head slots of a kv head rounded up to 4 or 8 (softmax lane layout).  SCORES: write the scaled scores only.
template <typename T, bool SCORES, int RK, int GP>
__global__ __launch_bounds__(512) void recon_spec_kernel(const FastParams p, const FactorOperand kB) {
  typedef typename Elem<T>::vec8 vec8;
  typedef SpecShape<RK> S;
  constexpr int FROW = S::FROW, FTILE = S::FTILE, NK = S::NK, NMB = S::NMB, SP_FLOATS = S::SP_FLOATS;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n32 = lane & 31, g2 = lane >> 5;
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
  const int ntiles = (end - start + FT - 1) / FT;
  const int nfull = (end - start) / FT;
  const int NPER = (ntiles + 2 + SRING - 1) / SRING * SRING;   // periods (one barrier each); the last tile's P.A runs in period ntiles + 1

  // ---- LDS carve-up ---------------------------------------------------------------------------------------------
  unsigned char* ring = smem;                                              // SRING * FTILE
  float* s_part = reinterpret_cast<float*>(smem + SRING * FTILE);          // [2][4 reconstruction waves][8 heads][FSP_ROW]
  sc_t* qhat = reinterpret_cast<sc_t*>(s_part + 2 * SP_FLOATS);            // [2][8 heads][128]
  sc_t* qzero = qhat + 2 * 8 * 128;                                        // [128] zeros: the q-dot operand of masked lanes
  float* unscale = reinterpret_cast<float*>(qzero + 128);                  // [8]
  const unsigned ring_lds = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)ring;

  // the factor, brought by all waves through the slot that no first tile is on its way to, and the scores behind it
  typedef FactorRows<T, RK> Factor;
  static_assert(FTILE + 2 * SP_FLOATS * 4 >= Factor::BYTES, "room for two chunks");
  Factor factor;
  const T* const Bh = reinterpret_cast<const T*>(kB.p) + b * kB.sb + kh * kB.sh;
  T* const stage = reinterpret_cast<T*>(ring + (SRING - 1) * FTILE);

  if (wave < 4) {
    // =================================================================================================================
    // reconstruction wave
    // =================================================================================================================
    float freq[8];         // of this lane's pairs 16 wave + 8 (r / 4) + 4 g2 + r % 4
#pragma unroll
    for (int r = 0; r < 8; ++r) freq[r] = p.inv_freq[16 * wave + 8 * (r >> 2) + 4 * g2 + (r & 3)];
    // ---- tile loads, straight to the LDS: rows 8 wave .. + 7 of a tile belong to this wave, one (RK * 2 bytes: lanes 0 .. RK/8 - 1) per
    // instruction.  Rows past the split's end are out of the resource's range and leave zeros; the softmax masks them.
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
    static_for<SRING - 1>([&](auto t_c) {
      next_tile();
      static_for<8>([&](auto r_c) { load_row(t_c, r_c); });
    });
    factor.template init<false>(Bh, kB.sr, tid);
    if (tid < 128) qzero[tid] = from_f32<sc_t>(0.f);
    // in-tile rotation of this wave's 8 pairs per lane (token n32, g2): pair 16 wave + 8 (r / 4) + 4 g2 + r % 4, r = 0 .. 7.  Two tables: the
    // query-side base is that of an EVEN tile and serves the odd tile after it too, whose offsets are 32 .. 63.
    float ct[2][8], st[2][8];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 8; ++r)
        __sincosf((float)(n32 + 32 * h) * freq[r], &st[h][r], &ct[h][r]);
    vec8 breg[NK];
    factor.pass(stage, tid, [&](int ch, const T* buf) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        breg[2 * ch + i] = Factor::operand(buf, 16 * i, wave, lane);
        asm volatile("" : "+a"(breg[2 * ch + i]));
      }
    });
    // q-dot B operand: lanes whose token half (lane bit 4) matches their column's (lane bit 3) read q^ of head lane % 8 (absent heads: the
    // last one; their columns are not used), the others read zeros
    const bool q_live = ((lane >> 4) & 1) == ((lane >> 3) & 1);
    const sc_t* qsrc = q_live ? qhat + ((lane & 7) < G ? (lane & 7) : G - 1) * 128 + ((wave & 1) * 4 + (wave >> 1)) * 16 + g2 * 8 : qzero;
    const int qpar = q_live ? 8 * 128 : 0;   // q^ is double-buffered by tile pair, the zeros are not
    float* const sdst = s_part + (wave * 8 + (n16 & 7)) * FSP_ROW + 16 * (n16 >> 3) + 4 * g4;
    f32x16 ka[2];          // two sets of key accumulators: registers 0 .. 7 the low features of the lane's pairs, 8 .. 15 their partners
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int r = 0; r < 16; ++r) ka[s][r] = 0.f;
    const unsigned char* fr0 = ring + n32 * FROW + 8 * g2 * 2;
    wait_vmcnt<0>();
    __syncthreads();        // tiles 0 to 2 are in the LDS, and the consumers' q^(0)

    // Period pp: the last LATE k-steps of tile pp-1 (accumulator set (pp-1) % 2; their operands were read before the barrier,
    // so the matrix pipe has work while the first operands of tile pp travel from the LDS), then the first NK - LATE k-steps
    // of tile pp (set pp % 2), with the rotation and the q-dot of tile pp-1 dealt out among them.
    // u = pp % 4 fixes every register and slot index at compile time.
    constexpr int LATE = S::LATE, EARLY = S::EARLY;
    vec8 carry[LATE];      // operands of the previous tile's last LATE k-steps
#pragma unroll
    for (int v = 0; v < LATE; ++v) carry[v] = ld16<vec8>(fr0 + v * 32);
    auto period = [&](int pp, auto u_c) {
      constexpr int u = decltype(u_c)::value, PAR = u & 1, SLOT = u % SRING;
      f32x16& k0 = ka[PAR];
      f32x16& j0 = ka[PAR ^ 1];
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) asm volatile("" : "+a"(breg[ks]));
      const unsigned char* fr = fr0 + SLOT * FTILE;
      // Rotation of tile pp-1 as 2 x 20 vector instructions, four pairs at a time, in three stages that depend on the stage before alone
      float tl[4], th[4], kl[4], kr[4];
      h2 kw[4];
      auto here = [](auto& v) { asm volatile("" : "+v"(v)); };   // computed at this place: without it the compiler sinks the chain to its end
      auto rotate = [&](auto u2_c) {
        constexpr int O = decltype(u2_c)::value / 20, U = decltype(u2_c)::value % 20, STAGE = U / 8, R = STAGE < 2 ? U % 8 / 2 : U - 16;
        const float lo = j0[4 * O + R], hi = j0[8 + 4 * O + R];
        const float cc = ct[PAR ^ 1][4 * O + R], ss = st[PAR ^ 1][4 * O + R];
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
      };
      // As the A operand of v_mfma_f32_16x16x32, lane (n32, g2) is row n32 % 16 and k-group (n32 / 16) + 2 g2; the B operand
      // keeps the token halves apart (column c' holds q^ of head c' % 8 in the k-groups of token half c' / 8, zeros elsewhere).
      // Result: lane (c', g4), register r = score of token 16 (c' / 8) + 4 g4 + r for head c' % 8.
      sc_vec8 qop[2];
      f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
      auto dot = [&](auto o_c) {
        const sc_vec8 kop = {kw[0][0], kw[0][1], kw[1][0], kw[1][1], kw[2][0], kw[2][1], kw[3][0], kw[3][1]};
        sacc = Elem<sc_t>::mfma16(kop, qop[decltype(o_c)::value], sacc);
      };
      // Past the last tile (and in period 0, which finishes a tile that does not exist) the same code runs on
      // whatever the LDS holds: nothing downstream uses those results, and one code path keeps the loop a single block.
      if (pp <= ntiles) {
        vec8 at[NK];
        constexpr int FIRST = LATE + 1, NROT = NK - 4 - FIRST;   // slots of the rotation
        constexpr int DOT0 = FIRST + (20 * NROT + 39) / 40, DOT1 = FIRST + NROT;
        static_for<NK>([&](auto v_c) {   // slot v of the period: one k-step
          constexpr int v = decltype(v_c)::value;
#pragma unroll
          for (int ks = 0; ks < NK; ++ks)
            if ((ks > EARLY ? ks - EARLY : 0) == v) at[ks] = ld16<vec8>(fr + ks * 32);   // read EARLY + LATE slots ahead of use
          if constexpr (v == LATE - 1) {
            const sc_t* qrow = qsrc + (((pp - 1) >> 1) & 1) * qpar;
            qop[0] = ld16<sc_vec8>(qrow);
            qop[1] = ld16<sc_vec8>(qrow + 32);
          }
          if constexpr (v < LATE) j0 = Elem<T>::mfma32(breg[NK - LATE + v], carry[v], j0);
          else if constexpr (v == LATE) {
            const f32x16 z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            k0 = Elem<T>::mfma32(breg[0], at[0], z);
          } else k0 = Elem<T>::mfma32(breg[v - LATE], at[v - LATE], k0);
          if constexpr (v == DOT0 + 1) dot(IC<0>());
          if constexpr (v == DOT1 + 1) dot(IC<1>());
          if constexpr (v >= FIRST && v < FIRST + NROT) {
            constexpr int U0 = (v - FIRST) * 40 / NROT, U1 = (v + 1 - FIRST) * 40 / NROT;
            static_for<U1 - U0>([&](auto i_c) { rotate(IC<U0 + decltype(i_c)::value>()); });
          }
          // the loads of tile pp + SRING - 1, spread evenly over the period: data that arrives in a burst keeps the LDS from the reads
          if constexpr (v == 0) next_tile();
          constexpr int LSTEP = NK / 8;
          if constexpr (v % LSTEP == LSTEP / 2) load_row(IC<(u + SRING - 1) % SRING>(), IC<v / LSTEP>());
          if constexpr (v == NK - 1) *reinterpret_cast<f32x4*>(sdst + (PAR ^ 1) * SP_FLOATS) = sacc;
          XKV_FENCE();
        });
#pragma unroll
        for (int v = 0; v < LATE; ++v) carry[v] = at[NK - LATE + v];
        wait_vmcnt<(SRING - 2) * 8>();   // this wave's rows of tile pp+1 have landed
      }
      __syncthreads();
    };
    for (int pb = 0; pb < NPER; pb += SRING) static_for<SRING>([&](auto u_c) { period(pb + decltype(u_c)::value, u_c); });
    wait_vmcnt<0>();
    return;
  }

  // ===================================================================================================================
  // consumer wave c
  // ===================================================================================================================
  const int c = wave - 4;

  // ---- query-side base rotation: thread -> pair j = lane, head slots c and c + 4 ------------------------------------------
  float q0[2], q1[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int h = c + 4 * i;
    if (h < G) {
      const T* qrow = reinterpret_cast<const T*>(p.q) + ((int64_t)b * p.hq + h0 + h) * 128;
      q0[i] = to_f32(qrow[lane]);
      q1[i] = to_f32(qrow[lane + 64]);
    } else {
      q0[i] = 0.f; q1[i] = 0.f;
    }
  }
  const float qinv = p.inv_freq[lane];
  factor.template init<false>(Bh, kB.sr, tid);
  {
    // Multiplied by the power of two that brings the head's largest feature to 2^14 .. 2^15, and the scores by the inverse: fp16 then holds every
    // rotated pair, and the parts of small queries are no subnormals there.  A feature that is no finite number leaves the others as they are.
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int bits = __builtin_bit_cast(int, row_reduce<true, 16>(fmaxf(fabsf(q0[i]), fabsf(q1[i]))));
      const int top = max(max(__builtin_amdgcn_readlane(bits, 0), __builtin_amdgcn_readlane(bits, 16)),
                          max(__builtin_amdgcn_readlane(bits, 32), __builtin_amdgcn_readlane(bits, 48)));
      const int up = max(-1, min(14 + 127 - (top >> 23), 100));
      const float f = __builtin_bit_cast(float, (127 + up) << 23);
      q0[i] *= f;
      q1[i] *= f;
      if (lane == 0) unscale[c + 4 * i] = __builtin_bit_cast(float, (127 - up) << 23);
    }
  }
  // q^ is kept in q-dot operand order: pair j = 32 dq' + 8 o + 4 g' + e sits at [o][dq'][g'][e] (partner at e + 4), so that
  // a lane's 8 contraction values of chunk o are one 16-byte read
  const int qpos = ((((lane >> 3) & 3) * 2 + (lane >> 5)) * 2 + ((lane >> 2) & 1)) * 8 + (lane & 3);
  float qc32, qs32, qcb, qsb;   // (qcb, qsb): base rotation of the tile whose q^ is written next
  sincosf((float)(2 * FT) * qinv, &qs32, &qc32);   // the base advances two tiles at a time
  // The base advances by angle addition and is replaced by a freshly range-reduced value every 30 tiles
  auto seed_qhat = [&](int t) { sincosf((float)(p.pos_offset + start + (int64_t)t * FT) * qinv, &qsb, &qcb); };
  seed_qhat(0);
  auto write_qhat = [&](int t) {   // q^ for the even tile t and the odd one after it = R(-base(t)) q, into buffer (t / 2) & 1
    sc_t* dst = qhat + ((t >> 1) & 1) * (8 * 128) + c * 128 + qpos;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (i == 1 && GP <= 4) break;   // head slots 4..7 are absent: nothing reads their rows
      dst[i * 512] = from_f32<sc_t>(q0[i] * qcb + q1[i] * qsb);
      dst[i * 512 + 4] = from_f32<sc_t>(q1[i] * qcb - q0[i] * qsb);
    }
    const float cc = qcb * qc32 - qsb * qs32, ss = qsb * qc32 + qcb * qs32;
    qcb = cc; qsb = ss;
  };
  write_qhat(0);
  factor.pass(stage, tid, [](int, const T*) {});

  // ---- softmax role: every consumer computes P of all heads; lane (n16, g4) holds head n16 % GP, tokens 8 g4 + TPL (n16 / GP) ..
  constexpr int TPL = GP / 2;   // tokens per lane
  const int sm_head = n16 & (GP - 1);
  const int sm_row = sm_head < G ? sm_head : G - 1;
  const int sm_tok = 8 * g4 + TPL * (n16 / GP);
  float m_ref = NEG_INF, l_run = 0.f;   // reference maximum of the lane's head (base-2 domain); this lane's share of its row sum
  const float lazy2 = lazy_rescale<T>() * 1.44269504088896f;
  // P.A accumulators (consumer c owns latent features RK/4 c .. + RK/4; column n16 = head slot) and the transposed tile reads
  // of two tiles live in accumulation registers a[0 .. 3 RK/16), by number (see pa_mfma_at)
  constexpr int TR0 = 4 * NMB, TRSET = 4 * NMB;
  static_for<4 * NMB>([&](auto r_c) { acc_set_at<decltype(r_c)::value>(0.f); });
  if constexpr (RK == 512) asm volatile("" ::: "a127");   // the kernel owns a[0 .. RK/4), which the reconstruction branch pins
  else if constexpr (RK == 384) asm volatile("" ::: "a95");
  else asm volatile("" ::: "a63");

  __syncthreads();
  const float scale2 = p.sm_scale * unscale[sm_row] * 1.44269504088896f;

  // Transposed reads: a 16-lane group reads a block of 4 rows x 16 columns, lanes 4 j .. 4 j + 3 supplying row j, and lane i
  // receives column i (4 values, one per row).  Rows 2 j (first read) and 2 j + 1 (second read) of the group's 8 tokens: with
  // the 16-byte row padding, rows two apart start 8 banks apart, so the 32-byte pieces of a read do not overlap (adjacent rows
  // would, by half).  Element e of the lane's 8 contraction values is therefore token 8 g4 + 2 e (e < 4) or 8 g4 + 2 (e - 4) + 1.
  const unsigned tr_base = ring_lds + (unsigned)((8 * g4 + 2 * (n16 >> 2)) * FROW + (c * (RK / 4) + 4 * (n16 & 3)) * 2);
  // softmax and P.A of tile t (partial scores in buffer t % 2, transposed tile in register set t % 2)
  typedef float fv __attribute__((ext_vector_type(TPL)));
  struct S23In { fv a[4]; };
  auto stage23_load = [&](auto tpar_c) {
    constexpr int TPAR = decltype(tpar_c)::value;
    S23In in;
    if (!SCORES) {
      const float* sp = s_part + TPAR * SP_FLOATS + sm_row * FSP_ROW + sm_tok;
#pragma unroll
      for (int w = 0; w < 4; ++w) in.a[w] = *reinterpret_cast<const fv*>(sp + w * 8 * FSP_ROW);
    }
    return in;
  };
  // (FULL: the tile lies wholly inside the split, no token is masked.)  The softmax runs in the base-2 domain: scores are
  // scaled by sm_scale * log2(e) in one multiplication and the reference maximum is kept in that domain, so that P is one
  // subtraction and one v_exp_f32 per score.
  auto stage23 = [&](int t, const S23In& in, auto ts_c, auto tpar_c, auto full_c) {
    constexpr int TS = decltype(ts_c)::value, TPAR = decltype(tpar_c)::value;
    constexpr bool FULL = decltype(full_c)::value != 0;
    if (SCORES) {   // consumer c writes heads c and c + 4: lane -> (head c + 4 (lane / 32), token lane % 32)
      const int head = c + 4 * g2;
      const float* sp = s_part + TPAR * SP_FLOATS + (head < G ? head : G - 1) * FSP_ROW + n32;
      const float s = ((sp[0] + sp[8 * FSP_ROW]) + (sp[2 * 8 * FSP_ROW] + sp[3 * 8 * FSP_ROW])) * (p.sm_scale * unscale[head]);
      const int tok = start + t * FT + n32;
      if (head < G && tok < end) {
        const int64_t o = ((int64_t)b * p.hq + h0 + head) * p.kv_len + tok;
        if (p.scores_dtype == XKV_F32) reinterpret_cast<float*>(p.scores)[o] = s;
        else reinterpret_cast<T*>(p.scores)[o] = from_f32<T>(s);
      }
      return;
    }
    float s[TPL];
    {
      const fv sum = (in.a[0] + in.a[1]) + (in.a[2] + in.a[3]);
#pragma unroll
      for (int e = 0; e < TPL; ++e) s[e] = sum[e];
    }
    const int tok = start + t * FT + sm_tok;
    float mxl = NEG_INF;
#pragma unroll
    for (int e = 0; e < TPL; ++e) {
      s[e] = (FULL || tok + e < end) ? s[e] * scale2 : NEG_INF;
      mxl = fmaxf(mxl, s[e]);
    }
    // the reference maximum only moves when the tile maximum exceeds it by the lazy bound; the cross-lane reduction that
    // finds the maximum runs only then.  Every consumer sees the same scores, so all four keep the same reference.
    if (__builtin_amdgcn_ballot_w64(mxl > m_ref + lazy2)) {   // rare: some head's maximum moves
      float mx = mxl;
#pragma unroll
      for (int m = GP; m < 64; m <<= 1) mx = fmaxf(mx, __shfl_xor(mx, m));
      const float m_new = mx > m_ref + lazy2 ? mx : m_ref;
      const float alpha = __builtin_amdgcn_exp2f(m_ref - m_new);
      m_ref = m_new;
      l_run *= alpha;
      if (__builtin_amdgcn_ballot_w64(alpha != 1.f)) {   // column n16 < GP of the accumulators is this lane's head
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        static_for<4 * NMB>([&](auto r_c) { acc_set_at<decltype(r_c)::value>(acc_get_at<decltype(r_c)::value>() * alpha); });
        asm volatile("s_nop 7" ::: "memory");
      }
    }
    float e[TPL];
    float esum = 0.f;
#pragma unroll
    for (int k = 0; k < TPL; ++k) {
      e[k] = __builtin_amdgcn_exp2f(s[k] - m_ref);
      esum += e[k];
    }
    l_run += esum;
    // P as the B operand of v_mfma_f32_16x16x32: lane (column n16 = head, g4) holds its head's tokens 8 g4 .. + 8 in the order
    // of the transposed reads (even tokens, then odd ones); lanes n16 < GP gather the other token groups of their head from
    // lanes n16 + GP, ... of the same 16-lane row (columns >= GP are unused)
    u32x4 pbu;
    if (GP == 4) {   // this lane: tokens 2 tq, 2 tq + 1; lane + 4: the next two
      const float y0 = __builtin_bit_cast(float, dpp_u32<0x104>(__builtin_bit_cast(unsigned, e[0])));
      const float y1 = __builtin_bit_cast(float, dpp_u32<0x104>(__builtin_bit_cast(unsigned, e[1])));
      const unsigned ev = pack_pair<T>(e[0], y0), od = pack_pair<T>(e[1], y1);   // (2 tq, 2 tq + 2), (2 tq + 1, 2 tq + 3)
      pbu = u32x4{ev, dpp_u32<0x108>(ev), od, dpp_u32<0x108>(od)};
    } else {         // this lane: tokens 4 tq .. + 4
      const unsigned ev = pack_pair<T>(e[0], e[TPL > 2 ? 2 : 0]), od = pack_pair<T>(e[1], e[TPL > 2 ? 3 : 1]);
      pbu = u32x4{ev, dpp_u32<0x108>(ev), od, dpp_u32<0x108>(od)};
    }
    static_for<NMB>([&](auto mb_c) {
      constexpr int mb = decltype(mb_c)::value;
      pa_mfma_at<T, 4 * mb, TR0 + TS * TRSET + 4 * mb>(pbu);
    });
  };

  // transposed reads of the tile in ring slot SLOT into register set TS; completion is awaited before the period's barrier
  auto trread = [&](auto ts_c, auto slot_c) {
    constexpr int TS = decltype(ts_c)::value, SLOT = decltype(slot_c)::value;
    const unsigned vt = tr_base + (unsigned)SLOT * FTILE;
    static_for<NMB>([&](auto mb_c) {
      constexpr int mb = decltype(mb_c)::value;
      tr_read_at<TR0 + TS * TRSET + 4 * mb, mb * 32>(vt);
      tr_read_at<TR0 + TS * TRSET + 4 * mb + 2, mb * 32 + FROW>(vt);
    });
  };

  // STEADY: tiles pp-2 .. pp+3 all exist and lie wholly inside the split.  Otherwise only the softmax + P.A step is
  // guarded (it must not touch its state for a tile that does not exist); the other steps run on whatever the LDS holds
  // and nothing uses their results.
  auto period = [&](int pp, auto u_c, auto steady_c) {
    constexpr int u = decltype(u_c)::value;
    constexpr bool STEADY = decltype(steady_c)::value != 0;
    const int t_pv = pp - 2;
    const bool pv_live = STEADY || (t_pv >= 0 && t_pv < ntiles);
    if (STEADY || pp < ntiles + 2) {
      const S23In in23 = stage23_load(IC<u & 1>());
      XKV_FENCE();
      if (pv_live) stage23(t_pv, in23, IC<u & 1>(), IC<u & 1>(), steady_c);
      XKV_FENCE();
      if (!SCORES) trread(IC<u & 1>(), IC<u % SRING>());
      XKV_FENCE();
      if ((u & 1) == 0 && pp >= 2) write_qhat(pp);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the transposed reads
    }
    __syncthreads();
  };
  for (int pb = 0; pb < NPER; pb += SRING) {
    if (pb > 0 && pb % 28 == 0) seed_qhat(pb);   // period pb writes q^ of tile pb next
    if (pb >= SRING && pb + 2 * SRING - 2 < nfull) static_for<SRING>([&](auto u_c) { period(pb + decltype(u_c)::value, u_c, IC<1>()); });
    else static_for<SRING>([&](auto u_c) { period(pb + decltype(u_c)::value, u_c, IC<0>()); });
  }
  if (SCORES) return;

  // ---- epilogue: every consumer holds every head's (reference, row sum); it normalises and writes its RK / 4 features ---------
  float l_head = l_run;
#pragma unroll
  for (int m = GP; m < 64; m <<= 1) l_head += __shfl_xor(l_head, m);
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  f32x4 acc[NMB];
  static_for<4 * NMB>([&](auto r_c) { constexpr int r = decltype(r_c)::value; acc[r >> 2][r & 3] = acc_get_at<r>(); });
  if (n16 < G) {
    const float inv = 1.f / l_head;
    const int64_t ph = ((int64_t)b * p.hq + h0 + n16) * p.max_splits + split;
    float* dst = p.partial + ph * RK + c * (RK / 4) + 4 * g4;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) *reinterpret_cast<f32x4*>(dst + mb * 16) = acc[mb] * inv;
    if (c == 0 && g4 == 0) p.lse[ph] = m_ref * 0.6931471805599453f + __logf(l_head);
  }
}

template <typename T, int RK>
int launch_recon_spec_t(const FastParams& p, const FactorOperand& kB, int batch, hipStream_t st) {
  typedef SpecShape<RK> S;
  const bool gp4 = p.hq / p.hkv <= 4;
  auto kern = p.scores ? (gp4 ? recon_spec_kernel<T, true, RK, 4> : recon_spec_kernel<T, true, RK, 8>)
                       : (gp4 ? recon_spec_kernel<T, false, RK, 4> : recon_spec_kernel<T, false, RK, 8>);
  static DynLds lds[4];
  const int e = ensure_dynamic_lds(lds[(p.scores ? 2 : 0) + (gp4 ? 1 : 0)], reinterpret_cast<const void*>(kern), (int)S::SHM, true);
  if (e != XKV_OK) return e;
  const int total = batch * p.hkv * p.max_splits;
  kern<<<dim3(xcd_grid(total, p.hkv)), dim3(512), S::SHM, st>>>(p, kB);
  return launch_status();
}

template <int RK>
int launch_recon_spec_rank(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st) {
  return dtype == XKV_BF16 ? launch_recon_spec_t<__bf16, RK>(p, kB, batch, st) : launch_recon_spec_t<_Float16, RK>(p, kB, batch, st);
}

}  // namespace spec
}  // namespace xkv
