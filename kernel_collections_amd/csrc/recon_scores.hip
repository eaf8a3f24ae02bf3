// Scores of rotated reconstructed keys:  K = kA @ kB[kh]  ->  rotate-half RoPE  ->  q . K'  ->  [batch, hq, kv_len].
//
// A wave holds the factor of a kv head for up to 256 ranks (rank x 128 x 2 bytes: 64 KB at 256) in its accumulation registers and
// rebuilds 16 tokens by itself: no partial keys to hand over.  Rotation and q-dot are linear in the key, so above 256 ranks two waves take
// half of the ranks each, rotate and multiply what they have, and only their SCORES are added up (WPT 2).
//
// One workgroup owns one (batch, kv head, split); a step is one tile of 16 tokens for every wave (WPT 1) or pair of waves (WPT 2).  A
// wave's rows go straight to a ring of four tiles of its own in the LDS, whole cache lines in consecutive lanes; read from
// memory in operand order, neighbouring lanes are different rows, and the cache looks up four lines where one would do (0.71 us for the
// loads of a 64-token step alone at rank 192).  Chunks of 16 bytes are exchanged within a row so that the operand reads meet no bank twice.
//
// The 128 features are rebuilt on v_mfma_f32_16x16x32, 16 pairs (j, j + 64) at a time: while the matrix pipe works on one block of
// pairs the vector pipe rotates the one before, in fp32, and hands it, rounded to fp16, to the q-dot as its A operand.
//
// RoPE by angle addition: R(position) = R(first token of the step) R(place in the step).  The second factor is per-lane constants; the
// first is moved to the query, q^ = R(step)^T q, which the workgroup needs once for all its tokens: in every group of two steps the waves
// make the q^ of the next group (a pair per lane) and leave it in the LDS, as a high and a low fp16 part: the scores are then as exact as those
// of an unrotated query (2.1e-4 of their size against float64, all of it the keys' rounding to fp16).  At rank 256 it is one fp16 value
// (2.9e-4), for callers that give a workspace and with it the wave-specialised kernel's one value: a low part costs 4 - 8 % there.
//
// What bounds it: one wave per SIMD that issues everything in order, an instruction in 5 cycles at best, and the LDS.  At 256 ranks the 68 matrix
// instructions of a tile are 1088 cycles, a block of 16 pairs takes 400 with everything else, and a group's start (barrier, q^)
// 500 more.  A branch or a memory operation waited for on the spot costs such a wave its whole latency, so the groups are straight-line code: places
// written whether they are needed or not, stores dropped by the resource's bounds, the output's form a template parameter.
// us at 131072 tokens, 8 kv heads, 32 heads: rank 64 34.9, 128 45.8, 192 57.9, 224 64.8, 256 63.8, 320 100, 448 122 (384 102, level with the wave-specialised kernel from 32768 tokens on); with rows read in operand
// order, rotation of keys by base and place, and branches rank 64 47.5, 128 53.7, 192 63.9, 256 77.8, 384 117.  Two waves per SIMD with half the pairs each
// and a barrier per step: 38.8, 50.5, 59.7, 73.7, 105.
#include "recon_fast.h"
#include "xkv_common.h"
#include <type_traits>
#include <utility>

namespace xkv {
namespace {

typedef short s16x4s __attribute__((ext_vector_type(4)));
typedef short s16x8s __attribute__((ext_vector_type(8)));
typedef sc_t sc_vec2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
template <int V> using IC = std::integral_constant<int, V>;
template <int N, typename F> __device__ __forceinline__ void unrolled(F f) {
  [&]<int... I>(std::integer_sequence<int, I...>) { (f(IC<I>()), ...); }(std::make_integer_sequence<int, N>());
}

constexpr int GROUP = 2;             // steps between barriers: the waves make q^ of the next ones
constexpr int SLOTS = 4;             // tiles of a wave's ring: the next one and three on the way (the one in use is in registers)
constexpr int BLD = 128 + 8;         // LDS row of the factor, elements
constexpr int SEED = 16;             // steps between range-reduced base angles: a multiple of SLOTS
enum { TO_F32, TO_16, TO_16_ODD };   // scores as stored: fp32, 16 bits a whole dword at a time, 16 bits each on its own (rows of odd length)
constexpr int OUT = -1;              // lane offset that no resource reaches: the store is dropped

template <int NKS, int WPT> struct ScoresShape {
  static constexpr int RK = 32 * NKS, RANK = RK * WPT;           // ranks of a wave
  static constexpr int STEP = 64 / WPT;                          // tokens
  static constexpr bool LO = RANK != 256;                        // q^ has a low part
  static constexpr int ROW = RK * 2, TILE = 16 * ROW, RING = SLOTS * 4 * TILE;   // [slot][wave][16 rows]
  // behind the ring: scores that wait for the other wave's [2 GROUP steps][wave][lane], q^ [2 groups][GROUP steps][parts][head][QROW words]
  static constexpr int PART = WPT == 1 ? 0 : 2 * GROUP * 4 * 64 * 16, QROW = 64 + 4;
  // the start's: angles of the waves' tiles, then the factor, RK ranks at a time, over all but the first two slots
  static constexpr int START = 2 * 4 * TILE, TABLE = 4 * 16 * 64 * 2 * 4, FACTOR = RK * BLD * 2;
  static constexpr int qheads(int G) { return G <= 4 ? 4 : (G + 1) & ~1; }   // two waves turn two heads each whatever the number
  // what the scores of even and of odd heads are multiplied by, behind all
  static constexpr int unscale(int G) {
    const int loop = RING + PART + 2 * GROUP * (LO ? 2 : 1) * qheads(G) * QROW * 4, start = START + (TABLE > FACTOR ? TABLE : FACTOR);
    return loop > start ? loop : start;
  }
  static constexpr int shm(int G) { return unscale(G) + 16; }
};

// N 1 KB pieces of a tile, to consecutive places in the LDS: an instruction's offset moves both addresses, so voff[i] is 1024 i less than what
// is read.  Waited for by count; addresses beyond the resource leave zeros.
template <int N> __device__ __forceinline__ void rows_to_lds(u32x4 res, const unsigned* voff, unsigned lds) {
  if constexpr (N == 1)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(voff[0]), "s"(res) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %3, 0 offen lds\n\tbuffer_load_dwordx4 %2, %3, 0 offen offset:1024 lds"
                 ::"s"(lds), "v"(voff[0]), "v"(voff[1]), "s"(res) : "memory", "m0");
}
template <int N> __device__ __forceinline__ void rows_landed() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ u32x4 resource(const unsigned char* p, int bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return u32x4{(unsigned)__builtin_amdgcn_readfirstlane((unsigned)a), (unsigned)__builtin_amdgcn_readfirstlane((unsigned)(a >> 32) & 0xffff),
               (unsigned)__builtin_amdgcn_readfirstlane((unsigned)bytes), 0x00020000u};
}

template <typename T, int NKS, int WPT, int MODE>
__global__ __launch_bounds__(256, 1) void recon_scores_kernel(const FastParams p, const FactorOperand kB) {
  typedef typename Elem<T>::vec8 vec8;
  typedef T vec4 __attribute__((ext_vector_type(4)));
  typedef T vec2 __attribute__((ext_vector_type(2)));
  typedef ScoresShape<NKS, WPT> S;
  constexpr int STEP = S::STEP, QROW = S::QROW, ROW = S::ROW;
  constexpr bool LO = S::LO;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tw = wave / WPT, half = WPT == 1 ? 0 : wave % WPT;   // tile of a step, part of the ranks
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
  const int tok0 = start + 16 * tw;
  const int n = (end - start + STEP - 1) / STEP;   // steps, the same for all waves

  // ---- token rows.  Piece l of a tile is its chunks 64 l .. + 63; chunk c of row r comes from chunk c ^ turn(r) of the row ------------
  const int row_bytes = (int)p.sAl * 2;
  auto turn = [](int r) { return NKS % 2 ? (r >> 1) & 3 : r & 7; };
  unsigned voff[NKS];
#pragma unroll
  for (int l = 0; l < NKS; ++l) {
    const int at = 64 * l + lane, r = at / (4 * NKS), c = at % (4 * NKS);
    voff[l] = r * row_bytes + (c ^ turn(r)) * 16 - (l % 2) * 1024;
  }
  const unsigned ring_lds = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)smem + wave * S::TILE;
  const unsigned char* arow = reinterpret_cast<const unsigned char*>(p.kA) + (b * p.sAb + half * S::RK) * 2 + (int64_t)tok0 * row_bytes;
  int aleft = L - tok0;      // rows of the sequence from arow on
  u32x4 ares;
  auto next_tile = [&]() {
    const int have = aleft < 16 ? aleft : 16;
    ares = resource(arow, have > 0 ? (have - 1) * row_bytes + ROW : 0);
    arow += (int64_t)STEP * row_bytes;
    aleft -= STEP;
  };
  constexpr int PAIRS = (NKS + 1) / 2;
  auto fetch = [&](auto slot_c, auto pair_c) {   // pieces 2 P and 2 P + 1
    constexpr int P = decltype(pair_c)::value;
    rows_to_lds<2 * P + 1 < NKS ? 2 : 1>(ares, voff + 2 * P, ring_lds + decltype(slot_c)::value * 4 * S::TILE + 2048 * P);
  };
  auto fetch_tile = [&](auto slot_c) {
    next_tile();
    unrolled<PAIRS>([&](auto p_c) { fetch(slot_c, p_c); });
  };
  fetch_tile(IC<0>());
  fetch_tile(IC<1>());

  // ---- queries, a pair per lane ------------
  constexpr int HEADS = 8;   // of 16 at most: this wave turns heads wave / 2, + 2, ...
  vec2 qp[HEADS];
#pragma unroll
  for (int j = 0; j < HEADS; ++j) {
    const int h = (wave >> 1) + 2 * j;
    const T* src = reinterpret_cast<const T*>(p.q) + ((int64_t)b * p.hq + h0 + (h < G ? h : 0)) * 128 + lane;
    qp[j] = vec2{src[0], src[64]};
  }

  // ---- the factor, through the LDS into accumulation registers: lane (feature n16, g4) holds 8 consecutive ranks ------------
  vec8 rows[2 * NKS * WPT];   // on the way while the angles are computed
  {
    const T* Bh = reinterpret_cast<const T*>(kB.p) + b * kB.sb + kh * kB.sh + (int64_t)(tid >> 4) * kB.sr + (tid & 15) * 8;
#pragma unroll
    for (int i = 0; i < 2 * NKS * WPT; ++i) rows[i] = ld16<vec8>(Bh + (int64_t)(16 * i) * kB.sr);
  }
  // cos, sin of the 16 places of this wave's tile in a step, a pair per lane: products of the powers of two, whose angles are exact
  const float inv = p.inv_freq[lane];
  float cg, sg, tc[16], ts[16];
  sincosf((float)(GROUP * STEP) * inv, &sg, &cg);
  sincosf((float)(16 * tw) * inv, &ts[0], &tc[0]);
#pragma unroll
  for (int o = 1; o < 16; o *= 2) {
    float s, c;
    sincosf((float)o * inv, &s, &c);
#pragma unroll
    for (int e = 0; e < o; ++e) {
      tc[o + e] = tc[e] * c - ts[e] * s;
      ts[o + e] = ts[e] * c + tc[e] * s;
    }
  }
  float* table = reinterpret_cast<float*>(smem + S::START) + wave * (16 * 64 * 2);
#pragma unroll
  for (int o = 0; o < 16; ++o) *reinterpret_cast<float2*>(&table[(o * 64 + lane) * 2]) = make_float2(tc[o], ts[o]);
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
  // This wave's queries are multiplied by the power of two that brings their largest feature to 2^14 .. 2^15, and the scores by the inverse.  fp16
  // then holds every rotated pair, which may be 1.41 times as long as its larger feature, and the parts of small queries are no subnormals there.
  // A feature that is no finite number leaves the others as they are.
  float* unscale = reinterpret_cast<float*>(smem + S::unscale(G));   // of even heads, of odd heads
  {
    float m = 0.f;
    auto largest = [&](auto j_c) {
      constexpr int J = decltype(j_c)::value;
      m = fmaxf(m, fmaxf(fabsf(to_f32(qp[J][0])), fabsf(to_f32(qp[J][1]))));
    };
    largest(IC<0>());
    largest(IC<1>());
    if (G > 4) unrolled<HEADS - 2>([&](auto j_c) { largest(IC<decltype(j_c)::value + 2>()); });
    const int bits = __builtin_bit_cast(int, row_reduce<true, 16>(m));
    const int top = max(max(__builtin_amdgcn_readlane(bits, 0), __builtin_amdgcn_readlane(bits, 16)),
                        max(__builtin_amdgcn_readlane(bits, 32), __builtin_amdgcn_readlane(bits, 48)));
    const int up = max(-1, min(14 + 127 - (top >> 23), 100));
    const float f = __builtin_bit_cast(float, (127 + up) << 23);
    auto lift = [&](auto j_c) {
      constexpr int J = decltype(j_c)::value;
      qp[J] = vec2{from_f32<T>(to_f32(qp[J][0]) * f), from_f32<T>(to_f32(qp[J][1]) * f)};
    };
    lift(IC<0>());
    lift(IC<1>());
    if (G > 4) unrolled<HEADS - 2>([&](auto j_c) { lift(IC<decltype(j_c)::value + 2>()); });
    if (lane == 0) unscale[wave >> 1] = __builtin_bit_cast(float, (127 - up) << 23);
  }
#pragma unroll
  for (int j = 0; j < HEADS; ++j) asm volatile("" : "+v"(qp[j]));   // waited for here: in the loop it would be a wait for rows
  vec8 breg[NKS][8];
  T* factor = reinterpret_cast<T*>(smem + S::START);
#pragma unroll
  for (int part = 0; part < WPT; ++part) {
    __syncthreads();   // every wave has read its table, the first half of the ranks
#pragma unroll
    for (int i = 0; i < 2 * NKS; ++i) st16(factor + ((tid >> 4) + 16 * i) * BLD + (tid & 15) * 8, rows[part * 2 * NKS + i]);
    __syncthreads();
    if (half == part) {
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
        for (int cbk = 0; cbk < 8; ++cbk) {
          const T* src = factor + (32 * ks + 8 * g4 + (n16 >> 2)) * BLD + 16 * cbk + 4 * (n16 & 3);
          s16x4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4s*)src);
          s16x4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4s*)(src + 4 * BLD));
          breg[ks][cbk] = __builtin_bit_cast(vec8, (s16x8s)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
  }
  __syncthreads();   // the factor's place becomes that of the other slots, of the scores and of q^
  fetch_tile(IC<2>());
  fetch_tile(IC<3>());

  // ---- q^ of the steps i0 + wave, lane = pair: words of (low feature, partner), 16 bytes for a lane's four pairs of a block ----------
  unsigned* qhat = reinterpret_cast<unsigned*>(smem + S::RING + S::PART);
  const int qpart = S::qheads(G) * QROW, qstep = (LO ? 2 : 1) * qpart;
  float cb = 1.f, sb = 0.f;
  unsigned* qdst = qhat + (wave & 1) * qstep + (wave >> 1) * QROW + lane;
  auto seed = [&](int i0) { sincosf((float)(p.pos_offset + start + (int64_t)(i0 + (wave & 1)) * STEP) * inv, &sb, &cb); };
  auto advance = [&]() {
    const float c = cb * cg - sb * sg;
    sb = sb * cg + cb * sg;
    cb = c;
  };
  auto turn_query = [&](int i0) {
    unsigned* dst = qdst + (i0 & GROUP) * qstep;
    auto turn = [&](auto j_c) {
      constexpr int J = decltype(j_c)::value;
      const float q0 = to_f32(qp[J][0]), q1 = to_f32(qp[J][1]);
      const float r0 = q0 * cb + q1 * sb, r1 = q1 * cb - q0 * sb;
      const sc_vec2 hi = {from_f32<sc_t>(r0), from_f32<sc_t>(r1)};
      dst[2 * J * QROW] = __builtin_bit_cast(unsigned, hi);
      if constexpr (LO) {
        const sc_vec2 lo = {from_f32<sc_t>(r0 - to_f32(hi[0])), from_f32<sc_t>(r1 - to_f32(hi[1]))};
        dst[qpart + 2 * J * QROW] = __builtin_bit_cast(unsigned, lo);
      }
    };
    turn(IC<0>());
    turn(IC<1>());
    if (G > 4) unrolled<HEADS - 2>([&](auto j_c) { if ((wave >> 1) + 2 * (decltype(j_c)::value + 2) < G) turn(IC<decltype(j_c)::value + 2>()); });
  };
  seed(0);
  turn_query(0);
  // lane (head n16, g4): heads past the kv head's repeat its first; their scores are never written
  const unsigned* qlane = qhat + (n16 < G ? n16 : 0) * QROW + 4 * g4;
  sc_vec8 qb[2][LO ? 2 : 1];   // q^ of a block, [parity]
  auto read_query = [&](int i, auto pb_c) {
    constexpr int PB = decltype(pb_c)::value;
    const unsigned* src = qlane + (i & (2 * GROUP - 1)) * qstep + 16 * PB;
#pragma unroll
    for (int e = 0; e < (LO ? 2 : 1); ++e) qb[PB & 1][e] = ld16<sc_vec8>(src + e * qpart);
  };

  // ---- operand of the tile in use: lane (token n16, g4) holds ranks 32 ks + 8 g4 .. + 7.  Replaced piece by piece while the last block
  // of a tile is multiplied ---------------------------------------------------------------------------------------------
  vec8 at[NKS];
  const unsigned char* aeven = smem + wave * S::TILE + n16 * ROW + ((g4 ^ turn(n16)) * 16);
  const unsigned char* aodd = smem + wave * S::TILE + n16 * ROW + (((4 + g4) ^ turn(n16)) * 16);
  auto read_rows = [&](auto slot_c, auto ks_c) {
    constexpr int KS = decltype(ks_c)::value, SLOT = decltype(slot_c)::value * 4 * S::TILE;
    if constexpr (NKS % 2) at[KS] = ld16<vec8>(aeven + SLOT + 64 * KS);
    else at[KS] = ld16<vec8>((KS % 2 ? aodd : aeven) + SLOT + 128 * (KS / 2));
  };
  rows_landed<3 * NKS>();
  unrolled<NKS>([&](auto ks_c) { read_rows(IC<0>(), ks_c); });

  f32x4 k[2][2];           // [parity of the block][low | partner features]
  f32x4 s_cur = {0.f, 0.f, 0.f, 0.f}, s_done[GROUP];
  k[0][0] = k[0][1] = k[1][0] = k[1][1] = s_cur;
#pragma unroll
  for (int u = 0; u < GROUP; ++u) s_done[u] = s_cur;
#pragma unroll
  for (int e = 0; e < (LO ? 2 : 1); ++e) qb[0][e] = qb[1][e] = sc_vec8{0, 0, 0, 0, 0, 0, 0, 0};

  // ---- scores: lane (head n16, g4) writes tokens 4 g4 .. + 3 of a tile.  Tile i of this wave lies at out + i * out_step -------------
  constexpr int es = MODE == TO_F32 ? 4 : 2;
  unsigned char* out = reinterpret_cast<unsigned char*>(p.scores) + (((int64_t)b * p.hq + h0) * p.kv_len + tok0) * es;
  const int out_step = STEP * es;
  const int olane = n16 < G ? (n16 * p.kv_len + 4 * g4) * es : OUT;
  const float scale = p.sm_scale * unscale[n16 & 1];
  auto store_full = [&](int i, int at_lane, f32x4 s) {   // a tile that ends before the split does
    s *= scale;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(out + (int64_t)i * out_step, 0, 0x7fffffff, 0x00020000);
    if constexpr (MODE == TO_F32) {
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, s), r, at_lane, 0, 0);
    } else {
      const vec4 v = {from_f32<T>(s[0]), from_f32<T>(s[1]), from_f32<T>(s[2]), from_f32<T>(s[3])};
      if constexpr (MODE == TO_16) {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, at_lane, 0, 0);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) __builtin_amdgcn_raw_buffer_store_b16(bits_of(v[e]), r, at_lane == OUT ? OUT : at_lane + 2 * e, 0, 0);
      }
    }
  };
  auto store_last = [&](int i, f32x4 s) {
    const int t = tok0 + i * STEP + 4 * g4;
    if (n16 >= G || t >= end) return;
    s *= scale;
    const int64_t o = ((int64_t)b * p.hq + h0 + n16) * p.kv_len + t;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (t + r < end) {
        if constexpr (MODE == TO_F32) reinterpret_cast<float*>(p.scores)[o + r] = s[r];
        else reinterpret_cast<T*>(p.scores)[o + r] = from_f32<T>(s[r]);
      }
  };
  // WPT 2: scores of a tile wait for the start of the next group, when the other wave's are there
  auto part = [&](int i, int w) { return reinterpret_cast<f32x4*>(smem + S::RING) + (((i & (2 * GROUP - 1)) * 4 + w) * 64 + lane); };

  // The rotation of a block of pairs as 20 vector instructions in three stages that depend on the stage before alone.
  float tl[4], th[4], kl[4], kr[4];
  sc_vec2 kw[4] = {};
  auto here = [](auto& v) { asm volatile("" : "+v"(v)); };   // computed at this place: without it the compiler sinks the chain to its end
  auto rotate = [&](auto pb_c, auto u_c) {
    constexpr int PB = decltype(pb_c)::value, U = decltype(u_c)::value, STAGE = U / 8, R = STAGE < 2 ? U % 8 / 2 : U - 16;
    const f32x4 &lo = k[PB & 1][0], &hi = k[PB & 1][1];
    if constexpr (STAGE == 0) {
      if constexpr (U % 2 == 0) { tl[R] = hi[R] * si[PB][R]; here(tl[R]); }
      else { th[R] = lo[R] * si[PB][R]; here(th[R]); }
    } else if constexpr (STAGE == 1) {
      if constexpr (U % 2 == 0) { kl[R] = __builtin_fmaf(lo[R], ci[PB][R], -tl[R]); here(kl[R]); }
      else { kr[R] = __builtin_fmaf(hi[R], ci[PB][R], th[R]); here(kr[R]); }
    } else {
      kw[R] = sc_vec2{from_f32<sc_t>(kl[R]), from_f32<sc_t>(kr[R])};
      here(kw[R]);
    }
  };
  auto dot = [&](auto pb_c, auto part_c, f32x4 s) {   // lane (head n16, g4): tokens 4 g4 + r
    const sc_vec8 kop = {kw[0][0], kw[0][1], kw[1][0], kw[1][1], kw[2][0], kw[2][1], kw[3][0], kw[3][1]};
    return Elem<sc_t>::mfma16(kop, qb[decltype(pb_c)::value & 1][decltype(part_c)::value % (LO ? 2 : 1)], s);
  };
  // Block PB of the tile in use: its matrix instructions, one by one, with the rotation of the block before dealt out among
  // them, and the q-dot of the one before that in front.  A wave that issues in order has both pipes wait for each other if either's
  // instructions come in a burst.
  f32x4 s_out[2];   // on their way to memory
  auto block = [&](int i, auto u_c, auto pb_c) {
    constexpr int SLOT = decltype(u_c)::value, PB = decltype(pb_c)::value, PR = (PB + 3) % 4, PD = (PB + 2) % 4, N = 2 * NKS;
    constexpr int LOW = N > 4 ? 2 : 0;
    constexpr int FIRST = N > 8 ? 2 : N > 2 ? 1 : 0;   // the last key of the block before is still under way in the first slots
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
    s_cur = dot(IC<PD>(), IC<0>(), PD == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : s_cur);
    __builtin_amdgcn_sched_barrier(0);
    unrolled<N>([&](auto m_c) {
      constexpr int M = decltype(m_c)::value;
      if constexpr (M % 2 == 0) lo = Elem<T>::mfma16(breg[M / 2][PB], at[M / 2], lo);
      else hi = Elem<T>::mfma16(breg[M / 2][4 + PB], at[M / 2], hi);
      constexpr int U0 = M < FIRST ? 0 : (M - FIRST) * 20 / (N - FIRST), U1 = M < FIRST ? 0 : (M + 1 - FIRST) * 20 / (N - FIRST);
      unrolled<U1 - U0>([&](auto u_c) { rotate(IC<PR>(), IC<U0 + decltype(u_c)::value>()); });
      if constexpr (LO && M == LOW) s_cur = dot(IC<PD>(), IC<1>(), s_cur);   // not next to the high part's, which it adds to
      // q^ for the dots of the next blocks, after this block's, which frees the registers; a step's last two before the barrier behind it
      if constexpr (M == LOW && PB > 0) read_query(i, IC<PR>());
      if constexpr (M == LOW + 1 && PB == 3) read_query(i, IC<3>());
      // rows of tile i + 4 into the slot of tile i, which is in registers from the end of block 0 on
      constexpr int P0 = PB == 0 ? 0 : (PB - 1) * PAIRS / 3, P1 = PB == 0 ? 0 : PB * PAIRS / 3, EVERY = N / (P1 > P0 ? P1 - P0 : 1);
      if constexpr (P0 < P1 && M % EVERY == EVERY / 2 && M / EVERY < P1 - P0) fetch(u_c, IC<P0 + M / EVERY>());
      // the next tile's operand: its rows are older than those of tiles i + 2 and i + 3 and than what the blocks before have sent for
      if constexpr (PB == 3 && M == 1) rows_landed<2 * NKS + (2 * PAIRS / 3) * 2>();
      if constexpr (PB == 3 && M % 2 == 1) read_rows(IC<(SLOT + 1) % SLOTS>(), IC<M / 2>());
      // stores of the tiles i - 3 and i - 2, at the start of a group
      if constexpr (SLOT % GROUP == 0 && WPT == 1 && PB == 1 && M == 0) store_full(i - 3, i < 3 ? OUT : olane, s_out[0]);
      if constexpr (SLOT % GROUP == 0 && WPT == 1 && PB == 2 && M == 0) store_full(i - 2, i < 2 ? OUT : olane, s_out[1]);
      if constexpr (SLOT % GROUP == 0 && WPT == 2 && PB == 0 && M == 0) { s_out[0] = *part(i - 3 + half, 2 * tw); s_out[1] = *part(i - 3 + half, 2 * tw + 1); }
      if constexpr (SLOT % GROUP == 0 && WPT == 2 && PB == 1 && M == 0) store_full(i - 3 + half, i < 3 - half ? OUT : olane, s_out[0] + s_out[1]);
      __builtin_amdgcn_sched_barrier(0);
    });
    k[PB & 1][0] = lo;
    k[PB & 1][1] = hi;
  };
  auto step = [&](int i, auto u_c) {   // tile i of this wave, i % SLOTS == U; finishes tile i - 1
    constexpr int W = (decltype(u_c)::value + 1) % GROUP;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int cbk = 0; cbk < 8; ++cbk) asm volatile("" : "+a"(breg[ks][cbk]));
    next_tile();
    block(i, u_c, IC<0>());
    block(i, u_c, IC<1>());
    s_done[W] = s_cur;
    block(i, u_c, IC<2>());
    if constexpr (WPT == 2) *part(i - 1, wave) = s_done[W];   // i = 0: a slot that is written again before it is read
    block(i, u_c, IC<3>());
  };
  // The start of the group of steps from i on.  The barrier: every wave has written its q^ of this group and, last group, its scores;
  // it has read those whose places are written next (behind the last group a barrier of its own says so).
  auto group = [&]() {
    __syncthreads();
    if constexpr (WPT == 1) { s_out[0] = s_done[1]; s_out[1] = s_done[0]; }
  };
  int i = 0;
  for (; i + SLOTS <= n; i += SLOTS) {
    group();
    advance();
    turn_query(i + GROUP);
    step(i, IC<0>());
    step(i + 1, IC<1>());
    group();
    if ((i + SLOTS) % SEED == 0) seed(i + SLOTS);
    else advance();
    turn_query(i + SLOTS);
    step(i + 2, IC<2>());
    step(i + 3, IC<3>());
  }
  if (i < n) {
    group();
    advance();
    turn_query(i + GROUP);
    step(i, IC<0>());
    if (i + 1 < n) step(i + 1, IC<1>());
    if (i + 2 < n) {
      i += GROUP;
      group();
      step(i, IC<2>());
    }
  } else {
    i -= GROUP;
  }
  // what is left of tile n - 1, and the tiles from i - 1 on, which no group has stored
  auto dots = [&](auto pb_c) {
    s_cur = dot(pb_c, IC<0>(), s_cur);
    if constexpr (LO) s_cur = dot(pb_c, IC<1>(), s_cur);
  };
  dots(IC<2>());
  unrolled<20>([&](auto u_c) { rotate(IC<3>(), u_c); });
  dots(IC<3>());
  if constexpr (WPT == 1) {
    if (i > 0) store_last(i - 1, s_done[1]);
    if (i < n - 1) store_last(i, s_done[0]);
    store_last(n - 1, s_cur);
  } else {
    // the last tile may lie where the last group's start has read tile i - 3, with no barrier since (n even, from 6 on)
    __syncthreads();
    *part(n - 1, wave) = s_cur;
    __syncthreads();
    for (int t = (i > 0 ? i - 1 : 0) + half; t < n; t += 2) store_last(t, *part(t, 2 * tw) + *part(t, 2 * tw + 1));
  }
  rows_landed<0>();   // tiles past the end: none may arrive in a place that is another workgroup's by then
}

template <typename T, int NKS, int WPT, int MODE>
int launch_t(const FastParams& p, const FactorOperand& kB, int batch, hipStream_t st) {
  typedef ScoresShape<NKS, WPT> S;
  auto kern = recon_scores_kernel<T, NKS, WPT, MODE>;
  const int shm = S::shm(p.hq / p.hkv);
  static DynLds lds;
  const int e = ensure_dynamic_lds(lds, reinterpret_cast<const void*>(kern), shm, true);
  if (e != XKV_OK) return e;
  kern<<<dim3(xcd_grid(batch * p.hkv * p.max_splits, p.hkv)), dim3(256), shm, st>>>(p, kB);
  return launch_status();
}

template <typename T, int MODE>
int launch_mode(const FastParams& p, const FactorOperand& kB, int batch, int rank, hipStream_t st) {
  switch (rank) {
#define XKV_SCORES_RANK(N) case 32 * N: return launch_t<T, N, 1, MODE>(p, kB, batch, st);
    XKV_SCORES_RANK(1) XKV_SCORES_RANK(2) XKV_SCORES_RANK(3) XKV_SCORES_RANK(4) XKV_SCORES_RANK(5) XKV_SCORES_RANK(6) XKV_SCORES_RANK(7)
    XKV_SCORES_RANK(8)
#undef XKV_SCORES_RANK
#define XKV_SCORES_RANK(N) case 64 * N: return launch_t<T, N, 2, MODE>(p, kB, batch, st);
    XKV_SCORES_RANK(5) XKV_SCORES_RANK(7)
#undef XKV_SCORES_RANK
    default: return XKV_EUNSUPPORTED;
  }
}

template <typename T>
int launch(const FastParams& p, const FactorOperand& kB, int batch, int rank, hipStream_t st) {
  if (p.scores_dtype == XKV_F32) return launch_mode<T, TO_F32>(p, kB, batch, rank, st);
  return p.kv_len % 2 == 0 && (reinterpret_cast<uintptr_t>(p.scores) & 3) == 0 ? launch_mode<T, TO_16>(p, kB, batch, rank, st)
                                                                              : launch_mode<T, TO_16_ODD>(p, kB, batch, rank, st);
}

}  // namespace

bool recon_scores_serves(const FastParams& p, const void* kB, int64_t sBb, int64_t sBh, int64_t sBr, int rank) {
  if (((sBb | sBh | sBr) & 7) || (reinterpret_cast<uintptr_t>(kB) & 15)) return false;
  if (rank > 224 && p.hq / p.hkv > 8) return false;                  // the LDS
  if (rank > 256 && rank != 320 && rank != 448) return false;        // two equal halves; 384 and 512 are faster elsewhere
  // 32-bit lane offsets: 16 token rows, the score rows of 16 heads.  Rows that overlap would make offsets negative
  return p.sAl >= rank && p.sAl < (1 << 25) && (int64_t)(p.hq / p.hkv) * p.kv_len < (1 << 28);
}

int launch_recon_scores(const FastParams& p, const void* kB, int64_t sBb, int64_t sBh, int64_t sBr, int batch, int dtype, int rank,
                        hipStream_t st) {
  const FactorOperand f{kB, sBb, sBh, sBr};
  return dtype == XKV_BF16 ? launch<__bf16>(p, f, batch, rank, st) : launch<_Float16>(p, f, batch, rank, st);
}

}  // namespace xkv
