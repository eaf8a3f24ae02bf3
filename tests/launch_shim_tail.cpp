// launch_shim.cpp with the two joined launches of prefix + tail decode, which a library of the same ABI may lack.
#include "launch_shim.cpp"

FORWARD(xkv_absorb_q_tail, true, (const void* q, const void* B, void* hi, void* lo, int b, int hq, int hkv, int d, int r, int64_t s0, int64_t s1,
                                  int64_t s2, xkv_kv_operand K, xkv_kv_operand V, int len, int S, float* part, float* lse, float scale, float lc, int dt,
                                  void* stream), (q, B, hi, lo, b, hq, hkv, d, r, s0, s1, s2, K, V, len, S, part, lse, scale, lc, dt, stream))
FORWARD(xkv_merge_stage2_tail, false, (const float* part, const float* lse, void* out, const void* vB, int64_t v0, int64_t v1, int64_t v2, int d, int dt,
                                       int b, int hq, int hkv, int L, int S, int dv, const float* tp, const float* tl, int ts, int64_t o0, int64_t o1,
                                       void* stream), (part, lse, out, vB, v0, v1, v2, d, dt, b, hq, hkv, L, S, dv, tp, tl, ts, o0, o1, stream))
