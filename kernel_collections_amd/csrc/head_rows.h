// Plain keys and values of 2, 4 or 8 kv heads of 128, side by side in a token row: one workgroup for all heads of a split (latent_ring.hip, the keys
// as one row), or one per kv head (latent_stage1.hip).  The lines between them, for stage 1's dispatcher and the host layers that choose its splits.
#pragma once
#include <algorithm>
#include <cstdint>

namespace xkv {

// us a call per kv head / as a row, rows read from memory.  32 heads on 4, one length: 4000 tokens 11.7 / 12.7, 8000 12.8 / 14.6, 16000 16.1 / 17.0, 2 x 8000 15.6 / 16.4, 2 x
// 10000 17.6 / 16.9, 2 x 16000 21.6 / 20.7: its 16-token tiles take 0.7 us each, and a short call has a few of them for each workgroup whatever the splits.  16 on
// 4: 4000 11.5 / 12.1, 8000 12.4 / 13.3, 10000 14.4 / 13.8, 2 x 16000 21.3 / 19.6; 4 on 4: 8000 12.4 / 13.0, 10000 14.2 / 13.5; 32 on 2: 2000 9.9 / 10.1, 4000 10.6 / 11.0, 8000
// 11.8 / 12.2, 10000 13.8 / 13.5.  16 on 2: no line (500 tokens 9.5 / 8.8, 24000 15.2 / 14.7), but see below; 8 heads: always a row.  Several lengths, 32 on 4: per kv head
// without a plan, up to 64 blocks of 64 tokens in all (2 x 2000 11.7 / 12.2, 4 x 500 10.4 / 11.0); beyond, a plan kernel goes in front of it (3 x 1500 15.6 / 11.7).
inline bool head_rows_pay(int heads, int hq, int64_t batch, int64_t kv_len, bool ragged, bool planned) {
  if (planned || heads == 8 || (heads == 2 && hq <= 16)) return true;
  const int64_t blocks = batch * ((kv_len + 63) / 64);
  if (ragged) return heads == 2 || hq <= 16 || blocks > 64;
  return blocks > (heads == 4 && hq > 16 ? 256 : 128);
}

// Rows of 2 heads: tiles of 32 tokens, two of which cost less than the partial rows of twice as many splits (us with splits of 32 / 64 tokens, 16 heads:
// 8000 tokens 12.7 / 11.9, 2 x 4000 11.9 / 11.5, 4000 11.3 / 11.3, 1000 10.4 / 10.6)
inline int head_rows_floor(int heads, int64_t tokens, int floor) { return heads == 2 && tokens > 4096 ? std::max(floor, 64) : floor; }

}  // namespace xkv
