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
//   rank 256: 32768 31.9 / 34.8, 45000 39.1 / 39.1, 53000 41.4 / 40.6, 65536 47.8 / 45.4; 64 on 16, 22528 36.2 / 36.2; 12 on 12, 32768 43.1 / 37.9; 16 on 4, 102400 40.5 / 41.8, 122880 46.4 / 46.1 (from
//   102400 on all the same: two passes, which the one-head kernel is not as exact as, take 50 there)
//   two kv heads, one workgroup for both: nothing is left to share a row's way from memory with.  Rank 512, 262144 95.2 / 93.6, 393216 132 / 125; rank 384, 262144 78.8 / 76.4
//   scores alone: rank 512, 16384 21.7 / 22.8, 24000 29.2 / 29.4, 48000 50.4 / 48.0, 16 on 2, 200000 61.5 / 61.7; rank 384, 64 on 8, 24000 24.6 / 25.6, 48000 41.9 / 41.4
inline int64_t recon_heads_work(int rank, int hkv) {
  if (hkv == 2) return 458752;
  return rank == 512 ? 229376 : rank == 384 ? 294912 : hkv == 4 ? 409600 : 344064;
}

// Workgroups from which on a host layer plans for it: the chip three quarters full
constexpr int64_t RECON_HEADS_WORKGROUPS = 192;

// Time of `live` (sequence, split) pairs of `groups` workgroups each, on 8 XCDs of 32 CUs: 160 a full round; a round of half of the CUs takes 0.7 of it, under the power limit
inline int64_t recon_rounds(int64_t live, int groups) {
  const int64_t n = (live + 7) / 8 * groups, rest = n % 32;
  return n / 32 * 160 + (rest ? 64 + 3 * rest : 0);
}
// Splits that somebody else chose, the same for every sequence: a tile takes a workgroup of two heads 7/4 as long as one of one head (rank 512: 2755 clocks and 1577), of four three
// times, so it is the last round that decides.  us of stage 1, several heads / one, 32 heads on 8 kv heads: rank 512, 98304 tokens, 32 splits 126 / 101, 48 97 / 117, 64 89 / 104, 80 127 / 118, 96
// 108 / 109, 112 102 / 122; 16 x 32768, 2 splits 626 / 520, 3 501 / 588, 4 453 / 527, 5 590 / 574, 6 509 / 531; rank 256, 65536, 64 splits 60.5 / 49.9, 96 45.3 / 51.9, 128 39.6 / 55.5, 160
// 61.4 / 60.4, 192 54.9 / 65.7
inline bool recon_heads_pays(int rank, int hkv, int nh, int64_t batch, int64_t kv_len, int64_t max_splits) {
  if (batch * kv_len * hkv < recon_heads_work(rank, hkv)) return false;
  const int64_t blocks = (kv_len + 31) / 32, per = (blocks + max_splits - 1) / max_splits, live = batch * ((blocks + per - 1) / per);
  return recon_rounds(live, hkv / nh) * (nh == 2 ? 7 : 12) <= recon_rounds(live, hkv) * 4;
}

// Scores at rank 256 of up to eight heads a kv head, by recon_scores_kernel or by one head a workgroup of the wave-specialised kernel, whose workgroups start faster, the more
// so the fewer kv heads read the same factor.  us a call, wave-specialised / recon_scores, 32 heads on 8 unless said: 1000 tokens 6.5 / 8.7, 12288 12.7 / 13.1, 16384 14.8 / 14.3, 32768
// 22.5 / 20.0; 16 on 4, 16384 9.2 / 10.3, 32768 13.1 / 13.1, 65536 21.2 / 19.6; 12 on 3, 43000 13.4 / 14.3, 54000 17.3 / 16.3; 16 on 2, 65536 14.1 / 15.3, 98304 18.4 / 18.3, 131072 22.5 /
// 21.4; 8 on 1, 131072 16.1 / 20.5, 524288 45.8 / 48.7, 8 x 16384 16.1 / 20.4, 2000000 229 / 230.  Rank 384 never: 32 on 8, 32768 28.4 / 28.3; 12 on 3, 130001 43.8 / 47.7; 4 on 1, 196608
// 27.6 / 29.7, 262144 34.1 / 36.7, 524288 82.4 / 84.9
inline bool recon_scores_pays(int rank, int hkv, int G, int64_t tokens) {
  return rank == 256 && G <= 8 && hkv > 1 && tokens * hkv >= (hkv == 2 ? 196608 : hkv == 3 ? 143360 : 131072);
}

}  // namespace xkv
