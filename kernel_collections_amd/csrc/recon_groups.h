// kv heads that a workgroup of recon_heads_kernel (recon_heads_impl.h) serves, and from which size on, for stage 1's dispatcher and the host layers that
// choose its splits.
#pragma once
#include <cstdint>

namespace xkv {

// 0: the kernel is not built for the shape.  Accumulation registers hold the factors: two heads of rank 512 or four of 256.  Scores of rank 256 stay with
// recon_scores_kernel (4 x 131072 tokens, 32 heads on 8: 236 / 242 us)
inline int recon_heads(int rank, int hkv, int G, bool scores) {
  if ((rank == 512 || rank == 384) && hkv % 2 == 0 && G <= 8) return 2;
  if (rank == 256 && !scores && hkv % 4 == 0 && G <= 4) return 4;
  return 0;
}

// Tokens x kv heads from which on host layers plan for it: a workgroup reads two or four factors before it starts, and has a half or a quarter of the tokens
// of one for one head.  us a call, one head a workgroup (recon_spec_kernel) / several, 32 heads on 8 kv heads unless said.
//   rank 512: 4096 tokens 24.4 / 25.3, 8192 28.1 / 28.4, 12000 31.9 / 30.9, 24000 42.1 / 40.1; 16 on 4, 2 x 12000 31.4 / 31.0; 64 on 8, 12000 33.4 / 33.4
//   rank 384: 8192 23.6 / 25.1, 16384 29.6 / 29.7, 24000 35.2 / 34.3; 16 on 4, 2 x 12000 26.2 / 27.5, 32768 30.8 / 30.2
//   rank 256: 16384 24.5 / 27.5, 24000 28.9 / 30.2, 32768 33.5 / 33.4, 48000 41.7 / 40.2; 16 on 4, 32768 25.9 / 28.3, 65536 34.6 / 34.5
//   two kv heads, one workgroup for both: nothing is left to share a row's way from memory with.  Rank 512, 66000 36.8 / 39.5, 131072 57.6 / 58.5, 262144 92.4 / 88.8; rank 384, 66000
//   32.1 / 33.3, 131072 47.4 / 46.6, 262144 78.0 / 73.9
//   scores alone: rank 512, 8192 15.7 / 15.6, 16384 22.8 / 21.8, 16 on 2, 66000 23.5 / 25.1, 131072 43.6 / 42.0; rank 384, 8192 13.3 / 13.2, 16384 18.9 / 18.2, 16 on 2, 66000 20.2 / 21.4
inline int64_t recon_heads_work(int rank, int hkv) {
  if (hkv == 2) return 327680;
  return rank == 512 ? 90112 : rank == 384 ? 131072 : 262144;
}

// Workgroups from which on the dispatcher takes it, whoever chose the splits: the chip three quarters full
constexpr int64_t RECON_HEADS_WORKGROUPS = 192;

}  // namespace xkv
