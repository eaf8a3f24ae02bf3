// The wave-specialised fused RoPE reconstruction kernel (recon_spec_impl.h) at rank 384.
#include "recon_spec_impl.h"

namespace xkv {

int launch_recon_spec_384(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st) {
  return spec::launch_recon_spec_rank<384>(p, kB, batch, dtype, st);
}

}  // namespace xkv
