// recon_heads_kernel at rank 256, four kv heads a workgroup.
#include "recon_heads_launch.h"

namespace xkv {

int launch_recon_heads_256(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st) {
  return heads::launch<false, 256, 4>(p, kB, batch, dtype, st);
}

}  // namespace xkv
