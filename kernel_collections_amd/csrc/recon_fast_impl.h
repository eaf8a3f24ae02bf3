// Pieces of the reconstruction kernels that read a tile for all ranks (recon_spec_impl.h, recon_heads_impl.h): direct-to-LDS row loads, tile constants.
#pragma once
#include "xkv_common.h"
#include "recon_fast.h"
#include <type_traits>
#include <utility>

namespace xkv {
namespace fast {

typedef short s16x4f __attribute__((ext_vector_type(4)));
typedef short s16x8f __attribute__((ext_vector_type(8)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int FT = 32;              // tokens per tile
constexpr int FSP_ROW = FT + 4;     // partial-score row stride (floats)
// The softmax reference only moves when a tile maximum exceeds it by this much.  P = exp(s - reference) is stored in the
// operand type, so the bound must keep exp(bound) finite there: e^16 = 8.9e6 fits bf16's exponent range, but fp16 ends
// at 65504 = e^11.09, hence 8 (e^8 = 2981) for fp16.
template <typename T> constexpr float lazy_rescale() { return std::is_same<T, _Float16>::value ? 8.f : 16.f; }

template <int V> using IC = std::integral_constant<int, V>;
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

template <int... I, typename F> __device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
  (f(IC<I>()), ...);
}
template <int N, typename F> __device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(std::make_integer_sequence<int, N>(), f);
}
template <int CTRL> __device__ __forceinline__ unsigned dpp_u32(unsigned x) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
}
template <typename T> __device__ __forceinline__ unsigned pack_pair(float a, float b) {
  typedef T t2 __attribute__((ext_vector_type(2)));
  const t2 v = {from_f32<T>(a), from_f32<T>(b)};
  return __builtin_bit_cast(unsigned, v);
}
// One row of a tile to the LDS.  Rows narrower than 1 KiB leave the lanes behind them out (their zeros would land in the next row); the wave
// runs with all lanes before and after.
template <int RK, int OFF> __device__ __forceinline__ void row_to_lds(u32x4 res, unsigned lane16, int row_off, unsigned lds) {
  unsigned at;
  if constexpr (RK == 512)
    asm volatile("s_add_u32 m0, %1, %5\n\tv_add_u32 %0, %2, %3\n\tbuffer_load_dwordx4 %0, %4, 0 offen lds"
                 : "=&v"(at) : "s"(lds), "s"(row_off), "v"(lane16), "s"(res), "n"(OFF) : "memory", "m0", "scc");
  else
    asm volatile("s_add_u32 m0, %1, %5\n\tv_add_u32 %0, %2, %3\n\ts_mov_b64 exec, %6\n\tbuffer_load_dwordx4 %0, %4, 0 offen lds\n\ts_mov_b64 exec, -1"
                 : "=&v"(at) : "s"(lds), "s"(row_off), "v"(lane16), "s"(res), "n"(OFF), "s"((1ull << (RK / 8 % 64)) - 1) : "memory", "m0", "scc");
}
template <int N> __device__ __forceinline__ void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

#define XKV_FENCE() __builtin_amdgcn_sched_barrier(0)

}  // namespace fast
}  // namespace xkv
