// Pieces of the wave-specialised reconstruction kernel (recon_spec_impl.h): direct-to-LDS row loads, the packed factor, tile constants.
#pragma once
#include "xkv_common.h"
#include "recon_fast.h"
#include <type_traits>

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

// The LDS destination of a direct-to-LDS load is M0 + lane * 16.  A SALU write of M0 needs one wait state
// before an instruction that reads M0 (the compiler schedules around this for its own code; here it is explicit).
// Address = scalar row base + per-lane byte offset.
__device__ __forceinline__ void async_row16(const void* row_base, unsigned lane_off, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(lane_off), "s"(row_base)
               : "memory", "m0");
}
// The instruction offset moves the LDS address AND the global address: with base = (first row of a group of four) - 128
// bytes and per-row lane offsets voff[r] = lane * 16 + 128 + r * (row_bytes - FROW), the instruction offset r * FROW puts
// global row r at tile row r, so the four rows of a group share one scalar base and one M0 value.  (FROW must stay below
// 4096 / 3 for the 13-bit offset field.)
template <int OFF>
__device__ __forceinline__ void async_row_off(const void* base_m128, unsigned voff, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3"
               ::"s"(lds_addr), "v"(voff), "s"(base_m128), "n"(OFF) : "memory", "m0");
}
template <int N> __device__ __forceinline__ void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// ---------------------------------------------------------------------------------------------------------------
// kB [hkv][RK][128] (strided) -> Bp [hkv][wave 4][ks RK/32][blk 2][lane 64][8]: the 16-byte packet lane l of wave
// (kq, dq) feeds to MFMA (ks, blk) as the A operand: B[RK/2 kq + 16 ks + 8 (l / 32) + e][64 blk + 32 dq + l % 32].
// ---------------------------------------------------------------------------------------------------------------
template <typename T, int RK>
__global__ __launch_bounds__(256) void pack_b_kernel(const T* __restrict__ kB, T* __restrict__ Bp, int64_t sBb, int64_t sBh,
                                                      int64_t sBr, int hkv) {
  const int kh = blockIdx.x, b = blockIdx.y;
  const T* Bh = kB + b * sBb + kh * sBh;
  constexpr int NKS = RK / 32;
  T* out = Bp + ((int64_t)b * hkv + kh) * (RK * 128);
  for (int idx = blockIdx.z * 256 + threadIdx.x; idx < 4 * NKS * 2 * 64; idx += 256 * gridDim.z) {
    const int l = idx & 63, blk = (idx >> 6) & 1, ks = (idx >> 7) % NKS, w = idx / (128 * NKS);
    const int kq = w >> 1, dq = w & 1;
    const int col = 64 * blk + 32 * dq + (l & 31);
    const int row0 = (RK / 2) * kq + 16 * ks + 8 * (l >> 5);
    typename Elem<T>::vec8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = Bh[(int64_t)(row0 + e) * sBr + col];
    st16(out + (int64_t)idx * 8, v);
  }
}

template <int V> using IC = std::integral_constant<int, V>;
#define XKV_FENCE() __builtin_amdgcn_sched_barrier(0)

}  // namespace fast
}  // namespace xkv
