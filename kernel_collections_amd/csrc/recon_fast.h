// Interface between the recon stage-1 dispatcher and its MFMA-bound paths (recon_scores.hip, recon_spec_*.hip, recon_duo_*.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace xkv {

struct FastParams {
  const void* q; const void* kA;
  int64_t sAb, sAl;
  float* partial; float* lse;
  void* scores; int scores_dtype;               // scores != NULL: write [batch, hq, kv_len] scaled scores, no softmax / P.A
  const int32_t* num_splits; const int32_t* kv_lens;
  int hq, hkv, kv_len, max_splits, total_wg;
  float sm_scale;
  const float* inv_freq; int64_t pos_offset;
  const void* vA; int64_t sVb, sVl;             // separate value basis (recon_duo kernels only)
};

struct FactorOperand { const void* p; int64_t sb, sh, sr; };   // kB [batch, hkv, rank, 128] in 16-byte packets

// The wave-specialised 8-wave kernel (recon_spec_impl.h), one translation unit per key rank: the key basis reused as
// the value basis, and the scores only that recon_scores.hip is not dispatched for (up to eight query heads per kv head).
int launch_recon_spec_512(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st);
int launch_recon_spec_384(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st);
int launch_recon_spec_256(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st);
inline int launch_recon_spec(const FastParams& p, const FactorOperand& kB, int batch, int dtype, int rank, hipStream_t st) {
  return rank == 512   ? launch_recon_spec_512(p, kB, batch, dtype, st)
         : rank == 384 ? launch_recon_spec_384(p, kB, batch, dtype, st)
                       : launch_recon_spec_256(p, kB, batch, dtype, st);
}

// Several kv heads per workgroup (recon_heads_impl.h): the shapes of recon_heads (recon_groups.h).
int launch_recon_heads_512(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st);
int launch_recon_heads_384(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st);
int launch_recon_heads_256(const FastParams& p, const FactorOperand& kB, int batch, int dtype, hipStream_t st);
inline int launch_recon_heads(const FastParams& p, const FactorOperand& kB, int batch, int dtype, int rank, hipStream_t st) {
  return rank == 512   ? launch_recon_heads_512(p, kB, batch, dtype, st)
         : rank == 384 ? launch_recon_heads_384(p, kB, batch, dtype, st)
                       : launch_recon_heads_256(p, kB, batch, dtype, st);
}

// Scores only (recon_scores.hip): ranks up to 224 with up to 16 query heads per kv head, 256, 320 and 448 with up to 8.  Reads kB as it is
// (16-byte packets of unit stride).
bool recon_scores_serves(const FastParams& p, const void* kB, int64_t sBb, int64_t sBh, int64_t sBr, int rank);
int launch_recon_scores(const FastParams& p, const void* kB, int64_t sBb, int64_t sBh, int64_t sBr, int batch, int dtype, int rank,
                        hipStream_t st);

// The 8-wave kernels (recon_duo_impl.h): key ranks 256 / 384 / 512 with a separate value basis of rank rv
inline bool recon_duo_serves(int rk, int rv) { return rv == rk || (rv == 512 && (rk == 384 || rk == 256)); }
int launch_recon_duo_b(const FastParams& p, const FactorOperand& kB, int batch, int dtype, int rk, int rv, hipStream_t st);   // 512 and 384
int launch_recon_duo_c(const FastParams& p, const FactorOperand& kB, int batch, int dtype, int rk, int rv, hipStream_t st);   // 256

}  // namespace xkv
