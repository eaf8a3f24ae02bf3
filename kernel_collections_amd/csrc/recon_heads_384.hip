// recon_heads_kernel at rank 384, two kv heads a workgroup.
#include "recon_heads_launch.h"

namespace xkv {

int launch_recon_heads_384(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st) {
  return p.scores ? heads::launch<true, 384, 2>(p, kB, batch, dtype, st) : heads::launch<false, 384, 2>(p, kB, batch, dtype, st);
}

}  // namespace xkv
