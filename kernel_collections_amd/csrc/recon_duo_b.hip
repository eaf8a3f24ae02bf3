// Shapes of the 8-wave fused RoPE reconstruction kernel built in this translation unit: separate value basis, key rank / value rank 512 / 512, 384 / 512, 384 / 384.
#include "recon_duo_impl.h"

namespace xkv {

int launch_recon_duo_b(const FastParams& p, const FactorOperand& kB, int batch, int dtype, int rk, int rv, hipStream_t st) {
  using namespace duo;
#define XKV_DUO_CASE(RK, RV) \
  if (rk == RK && rv == RV) return launch_duo<RK, RV>(p, kB, batch, dtype, st);
  XKV_DUO_CASE(512, 512) XKV_DUO_CASE(384, 512) XKV_DUO_CASE(384, 384)
#undef XKV_DUO_CASE
  return XKV_EUNSUPPORTED;
}

}  // namespace xkv
