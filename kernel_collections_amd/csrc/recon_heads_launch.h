// Launches of recon_heads_kernel: one translation unit per key rank.
#pragma once
#include "recon_heads_impl.h"

namespace xkv {
namespace heads {

template <typename T, bool SCORES, int RK, int GP, int NH>
int launch_t(FastParams p, const FactorOperand& kB, int batch, hipStream_t st) {
  typedef HeadsShape<RK, NH, SCORES, NH * GP / 2> S;
  auto kern = recon_heads_kernel<T, SCORES, RK, GP, NH>;
  static DynLds lds;
  const int e = ensure_dynamic_lds(lds, reinterpret_cast<const void*>(kern), (int)S::SHM, true);
  if (e != XKV_OK) return e;
  p.total_wg = batch * (p.hkv / NH) * p.max_splits;
  kern<<<dim3(xcd_grid(p.total_wg, p.hkv / NH)), dim3(256), S::SHM, st>>>(p, kB);
  return launch_status();
}
// up to 16 / NH query heads per kv head
template <typename T, bool SCORES, int RK, int NH>
int launch_heads(const FastParams& p, const FactorOperand& kB, int batch, hipStream_t st) {
  if constexpr (NH == 2)
    if (p.hq / p.hkv > 4) return launch_t<T, SCORES, RK, 8, NH>(p, kB, batch, st);
  return launch_t<T, SCORES, RK, 4, NH>(p, kB, batch, st);
}
template <bool SCORES, int RK, int NH>
int launch(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st) {
  return dtype == XKV_BF16 ? launch_heads<__bf16, SCORES, RK, NH>(p, kB, batch, st) : launch_heads<_Float16, SCORES, RK, NH>(p, kB, batch, st);
}

}  // namespace heads
}  // namespace xkv
