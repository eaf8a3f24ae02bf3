// A kv head's factor [RK, 128] as it is in memory, to the A operands of v_mfma_f32_32x32x16 of a workgroup of 8 waves: whole rows in 16-byte packets to
// registers, through the LDS 32 rows at a time, back by transposed reads (in memory a rank is a row, the operand wants consecutive ranks in a lane).
//
// A launch in front that packed the factor in operand order took 2.6 us of a call of 20, all of it the latency of a launch and a round trip.  Here the rows arrive
// beside the first tiles, which take as long; the way through the LDS is RK / 32 barriers of some 100 ns.
#pragma once
#include "xkv_common.h"

namespace xkv {

template <typename T, int RK> struct FactorRows {
  typedef typename Elem<T>::vec8 vec8;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  static constexpr int CHUNKS = RK / 32, DEEP = CHUNKS < 8 ? CHUNKS : 8;   // DEEP: chunks on the way
  static constexpr int LD = 128 + 8;                                       // a row in the LDS
  static constexpr int BYTES = 2 * 32 * LD * 2;                            // two chunks in turn
  vec8 rows[DEEP];
  const T* src;
  int64_t step;
  // Chunk c: ranks 32 c .. + 32, or (HALVES) 16 c .. + 16 of both halves of the ranks.  Thread tid brings packet tid % 16 of row tid / 16.
  template <bool HALVES> __device__ __forceinline__ void init(const T* head, int64_t sr, int tid) {
    const int i = tid >> 4;
    src = head + (HALVES ? (i >> 4) * (RK / 2) + (i & 15) : i) * sr + (tid & 15) * 8;
    step = (HALVES ? 16 : 32) * sr;
#pragma unroll
    for (int c = 0; c < DEEP; ++c) rows[c] = ld16<vec8>(src + c * step);
  }
  // use(c, buffer): every wave's reads of chunk c
  template <typename Use> __device__ __forceinline__ void pass(T* stage, int tid, Use use) {
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      T* buf = stage + (c & 1) * 32 * LD;
      st16(buf + (tid >> 4) * LD + (tid & 15) * 8, rows[c % DEEP]);
      if (c + DEEP < CHUNKS) rows[c % DEEP] = ld16<vec8>(src + (c + DEEP) * step);
      __syncthreads();   // whoever is here has read the chunk before, whose place the next one takes
      use(c, buf);
    }
  }
  // Lane (feature 64 (n32 / 16) + 16 quarter + n16, g2): ranks 8 g2 .. + 8 of the 16 rows from `row` on
  static __device__ __forceinline__ vec8 operand(const T* buf, int row, int quarter, int lane) {
    const int n16 = lane & 15;
    const T* at = buf + (row + 8 * (lane >> 5) + (n16 >> 2)) * LD + 64 * ((lane >> 4) & 1) + 16 * quarter + 4 * (n16 & 3);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)at);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(at + 4 * LD));
    return __builtin_bit_cast(vec8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
};

}  // namespace xkv
