// Which kernel serves a call of generated angles at ranks 512, 384 and 256, from which size on: kv heads that a workgroup of recon_heads_kernel (recon_heads_impl.h)
// serves, and scores by recon_scores_kernel, for stage 1's dispatcher and the host layers that choose its splits.
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
//   rank 512: 12000 tokens 30.5 / 32.4, 20000 37.3 / 37.8, 24000 41.1 / 41.1, 32000 49.3 / 47.9; 16 on 4, 2 x 24000 40.9 / 41.4, 2 x 32768 49.1 / 48.1; 64 on 8, 24000 42.1 / 43.5
//   rank 384: 24000 34.1 / 35.2, 32768 40.5 / 40.7, 48000 52.3 / 51.4; 16 on 4, 32768 29.7 / 31.2, 65536 41.6 / 41.0
//   rank 256: 32768 32.6 / 34.0, 48000 41.4 / 40.8, 65536 51.8 / 47.5; 16 on 4, 65536 34.2 / 35.2, 131072 53.4 / 48.5
//   two kv heads, one workgroup for both: nothing is left to share a row's way from memory with.  Rank 512, 262144 95.2 / 93.6, 393216 132 / 125; rank 384, 262144 78.8 / 76.4
//   scores alone: rank 512, 16384 21.7 / 22.8, 24000 29.2 / 29.4, 48000 50.4 / 48.0, 16 on 2, 200000 61.5 / 61.7; rank 384, 64 on 8, 24000 24.6 / 25.6, 48000 41.9 / 41.4
inline int64_t recon_heads_work(int rank, int hkv) {
  if (hkv == 2) return 458752;
  return rank == 512 ? 229376 : rank == 384 ? 294912 : 344064;
}

// Workgroups from which on the dispatcher takes it, whoever chose the splits: the chip three quarters full
constexpr int64_t RECON_HEADS_WORKGROUPS = 192;

// Scores at rank 256 of up to eight heads a kv head, by recon_scores_kernel or by one head a workgroup of the wave-specialised kernel, whose workgroups start faster, the more
// so the fewer kv heads read the same factor.  us a call, wave-specialised / recon_scores, 32 heads on 8 unless said: 1000 tokens 6.5 / 8.7, 12288 12.7 / 13.1, 16384 14.8 / 14.3, 32768
// 22.5 / 20.0; 16 on 4, 16384 9.2 / 10.3, 32768 13.1 / 13.1, 65536 21.2 / 19.6; 12 on 3, 43000 13.4 / 14.3, 54000 17.3 / 16.3; 16 on 2, 65536 14.1 / 15.3, 98304 18.4 / 18.3, 131072 22.5 /
// 21.4; 8 on 1, 131072 16.1 / 20.5, 524288 45.8 / 48.7, 8 x 16384 16.1 / 20.4, 2000000 229 / 230.  Rank 384 never: 32 on 8, 32768 28.4 / 28.3; 12 on 3, 130001 43.8 / 47.7; 4 on 1, 196608
// 27.6 / 29.7, 262144 34.1 / 36.7, 524288 82.4 / 84.9
inline bool recon_scores_pays(int rank, int hkv, int G, int64_t tokens) {
  return rank == 256 && G <= 8 && hkv > 1 && tokens * hkv >= (hkv == 2 ? 196608 : hkv == 3 ? 143360 : 131072);
}

}  // namespace xkv
