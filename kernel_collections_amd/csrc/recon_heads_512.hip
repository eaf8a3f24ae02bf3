// recon_heads_kernel at rank 512, two kv heads a workgroup.
#include "recon_heads_launch.h"

namespace xkv {

int launch_recon_heads_512(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st) {
  return p.scores ? heads::launch<true, 512, 2>(p, kB, batch, dtype, st) : heads::launch<false, 512, 2>(p, kB, batch, dtype, st);
}

}  // namespace xkv
