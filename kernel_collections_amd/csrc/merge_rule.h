// Forms of the up-projecting merge (merge_up_kernel in small_kernels.hip), for its dispatcher and for the host layers that may merge the rows in a launch of their own first.
#pragma once
#include <cstdint>

namespace xkv {

constexpr int MERGE_CB = 64;       // columns per workgroup: whole 128-byte lines of a vB row

inline int64_t merge_blocks(int64_t heads, int64_t batch, int d_out) { return heads * batch * ((d_out + MERGE_CB - 1) / MERGE_CB); }

// Heads of a workgroup that folds a packet's splits in one thread: those of a kv head (vB is read once for them) as far as their merged rows fit 48 KiB of LDS
inline int merge_heads(int64_t hq, int hkv, int64_t dv, int64_t batch, int d_out) {
  const int g = (int)(hq / hkv);
  int hpw = g;
  while (hpw > 1 && (g % hpw != 0 || hpw * dv * 4 > 48 * 1024)) --hpw;
  while (hpw > 4 && hpw % 2 == 0 && merge_blocks(hq / hpw, batch, d_out) < 256) hpw /= 2;
  return hpw;
}

// One head a workgroup, its splits dealt out among groups of threads, where that is not more than a workgroup per CU (each reads its head's part of vB again) and a head
// has splits to deal out.  us, a graph of merges, 32 heads on 8 kv heads, d_out 128 unless said: a thread all splits / dealt out.  Batch 1, values of 256: 8 splits 4.5 / 4.9, 16 5.1 /
// 4.9, 32 6.3 / 4.9, 64 8.7 / 5.2; of 512: 8 6.1 / 5.8, 32 7.9 / 6.5, 128 18.1 / 9.5; 64 heads, 32 of 512 7.9 / 7.0; batch 4, 16 of 512 7.5 / 6.6; batch 8, 16 of 512 7.9 / 9.3; 16 on
// 1, d_out 512, batch 8, 32 of 256 7.0 / 9.3
inline bool merge_spread(int64_t splits, int64_t hq, int64_t batch, int64_t dv, int d_out) {
  return splits > 1 && splits * dv >= 4096 && merge_blocks(hq, batch, d_out) <= 256;
}

// One head a workgroup too where there is little to fold: all heads of a kv head / one, 32 on 8 heads unless said.  Batch 1, one row of 512 5.8 / 4.8, of 256 4.2 / 3.7, 4 splits of
// 512 6.0 / 4.8; 32 on 1, d_out 512, one of 512 5.9 / 4.9; batch 4, 7 splits of 512 6.3 / 5.1; batch 5, one of 512 5.9 / 6.6, batch 16 6.2 / 11.3
inline bool merge_one_head(int64_t hq, int64_t batch, int d_out) { return merge_blocks(hq, batch, d_out) <= 256; }

// Partial values that a workgroup may fold in every column block, of one head (dealt out) or of all of its heads; beyond, the rows are merged first, by the whole chip.  us of one kernel
// / rows and up-projection: dealt out, batch 1, 128 splits of 512 9.5 / 10.2, 256 of 256 8.6 / 9.7, 256 of 384 11.7 / 11.0, 16 on 2, 128 of 512 8.3 / 8.7
constexpr int64_t MERGE_FLOATS = 65536;
// Where a thread folds all splits of its packets one after another, every column block reads them again: out of the same XCD's L2 if the blocks of a head lie on one (workgroups go round-robin
// over the 8 XCDs, heads and sequences first), else from memory.  With more than 16 splits that decides earlier, and so do, of more than two blocks, a second round of workgroups and more than 48 splits.
// us of a whole call, one kernel / rows and up-projection, 512 columns.  On one XCD, 16 on 1, 6 sequences, 40 splits of 384 (61440 values) 30.4 / 31.8, 8, 30 of 512 (61440) 33.9 / 35.4, 4, 59 of 256
// (60416) 27.4 / 25.9; 32 on 1, 5, 47 of 256 (48128) by 0.7, 12, 20 of 256 (40960) by 1.6 one kernel, 7, 34 of 384 (52224) 36.6 / 35.8.  Apart, 16 on 1, 9, 27 of 256 (27648) 0.1, of 384 (41472)
// 36.2 / 34.2, 13, 19 of 384 (29184) 35.9 / 35.0, 7, 34 of 256 (34816) 26.9 / 26.3, of 384 33.0 / 31.8, 27, 9 of 512 (36864) 42.8 / 44.2, 17, 14 of 512 (57344) by 0.9 one kernel; 16 on 2, 128 columns, 9, 28 of 384 (43008) 46.9 / 46.4,
// 17, 14 of 512 (28672) 46.9 / 48.9
constexpr int64_t MERGE_FLOATS_APART = 28672, MERGE_FLOATS_ROUNDS = 49152;
inline bool merge_rows_first(int64_t splits, int64_t hq, int hkv, int64_t dv, int64_t batch, int d_out) {
  if (splits <= 1) return false;
  if (merge_spread(splits, hq, batch, dv, d_out)) return splits * dv > MERGE_FLOATS;
  const int hpw = merge_heads(hq, hkv, dv, batch, d_out);
  const int64_t values = splits * hpw * dv;
  if (splits <= 16) return values > MERGE_FLOATS;
  const bool apart = d_out > MERGE_CB && hq / hpw * batch % 8;
  if (apart) return values > MERGE_FLOATS_APART;
  const bool rounds = d_out > 2 * MERGE_CB && (splits > 48 || merge_blocks(hq / hpw, batch, d_out) > 256);
  return values > (rounds ? MERGE_FLOATS_ROUNDS : MERGE_FLOATS);
}

// The same with a tail's rows beside them (xkv_merge_stage2_tail), whose splits no form deals out: a thread folds all of a packet's.  The line counts all heads of a kv head also where a
// workgroup takes one (merge_one_head), for which it lies early: us of a call, 32 heads on one matrix, batch 1, rank 512, tail 128, one kernel / rows first, 8 splits 23.5 / 26.7, 16 24.5 / 27.1,
// 32 26.6 / 28.0, and 64, from 2048 tokens of prefix on, 30.8 / 29.4 (rank 256 22.0 / 21.0; 4 x 8 heads 26.3 / 25.0)
constexpr int64_t MERGE_TAIL_FLOATS = 49152;
inline bool merge_tail_rows_first(int64_t splits, int64_t hq, int hkv, int64_t dv) { return splits > 1 && splits * (hq / hkv) * dv > MERGE_TAIL_FLOATS; }

}  // namespace xkv
