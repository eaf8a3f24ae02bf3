"""Shared host logic of the fused xKV decode wrappers (no-PE, K-only, RoPE)."""
from __future__ import annotations

from typing import Optional

import torch

from kernel_collections_amd import _lib, ops


def _common(q, k_A, k_B):
    assert q.dim() == 3, "q must be [batch, num_q_heads, head_dim]"
    batch, num_q_heads, head_dim = q.shape
    num_kv_heads = k_B.shape[1]
    assert k_A.shape[0] == batch and k_B.shape[0] == batch, "Batch size mismatch"
    assert k_A.shape[-1] == k_B.shape[2], "Rank mismatch between k_A and k_B"
    assert k_B.shape[-1] == head_dim, "Head dimension mismatch"
    assert num_q_heads % num_kv_heads == 0
    kv_group_num = num_q_heads // num_kv_heads
    assert kv_group_num >= 1
    assert k_A.shape[-1] % 32 == 0, "rank must be a multiple of 32"
    return batch, num_q_heads, num_kv_heads, head_dim


def _lens(kv_lens, batch, device):
    return None if kv_lens is None else ops.as_int32_dev(kv_lens, batch, device)


def _plan(lens, batch, groups, kv_len, rank, absorbed=True, up=False):
    """(num_kv_splits, cap, split dimension, plan) that fill the device: the caller's count is a hint (split-K is exact under the
    merge), and 128 splits of one long sequence - the reference scripts' count - would leave half the CUs idle."""
    if lens is not None and batch > 1:
        per_cu = 1 if absorbed and rank in (256, 384, 512) else 2
        return ops.ragged_plan(lens, batch, groups, kv_len, ops.split_floor(batch, groups, kv_len, per_cu, up), per_cu)
    S = ops.latent_splits(batch, groups, kv_len, rank, absorbed=absorbed)
    return None, 0, S, None


def decode_nope(q, k_A, k_B, v_A, v_B, o, num_kv_splits, max_kv_splits, sm_scale, kv_lens=None):
    """K and V factorised, no positional encoding: absorb q into k_B, scan k_A / v_A once for
    all heads, merge in rank space, then multiply by v_B."""
    ops.check_splits(num_kv_splits, max_kv_splits, q.shape[0])
    native = _lib.native()
    done = native and native.nope_decode(q, k_A, k_B, v_A, v_B, o, sm_scale, kv_lens)
    if done is not None:
        return done
    assert v_A.shape[1] == k_A.shape[1]
    assert v_B.shape[1] == k_B.shape[1]
    batch, hq, hkv, d = _common(q, k_A, k_B)
    ops.check_16bit(q, k_A, k_B, v_A, v_B)
    rank_v = v_A.shape[-1]
    assert rank_v == v_B.shape[2], "Rank mismatch between v_A and v_B"
    assert rank_v % 64 == 0 and rank_v <= 512, "v rank must be a multiple of 64, at most 512"
    kv_len = k_A.shape[1]
    lens = _lens(kv_lens, batch, q.device)
    q3 = ops._q3(q)
    k_A, v_A = ops.as_rows(k_A), ops.as_rows(v_A)
    qt_hi, qt_lo = ops.absorb_q(q3, k_B, want_lo=True)
    groups = ops.head_groups(hq)
    splits, cap, S, plan = _plan(lens, batch, groups, kv_len, k_A.shape[-1], up=True)
    partial, lse = ops.workspaces(batch, hq, S, rank_v, q.device, plan)
    ops.latent_stage1(qt_hi, qt_lo, None, (k_A, k_A.stride(0), k_A.stride(1), 0, k_A.shape[-1]), None,
                      (v_A, v_A.stride(0), v_A.stride(1), 0, rank_v), partial, lse, None, splits, lens,
                      batch, hq, groups, kv_len, S, float(sm_scale), split_cap=cap, split_plan=plan)
    return ops.merge_stage2(partial, lse, o, v_B, splits, lens, batch, hq, hkv, kv_len, S, split_cap=cap, split_plan=plan)


def decode_k_only(q, k_A, k_B, v_buffer, o, num_kv_splits, max_kv_splits, sm_scale, kv_lens=None):
    """K factorised (absorbed), V plain ``[batch, kv_len, num_kv_heads, head_dim]``."""
    ops.check_splits(num_kv_splits, max_kv_splits, q.shape[0])
    batch, hq, hkv, d = _common(q, k_A, k_B)
    ops.check_16bit(q, k_A, k_B, v_buffer)
    assert v_buffer.shape[1] == k_A.shape[1] and v_buffer.shape[2] == hkv
    dv = v_buffer.shape[-1]
    assert dv % 64 == 0 and dv <= 512
    kv_len = k_A.shape[1]
    lens = _lens(kv_lens, batch, q.device)
    q3 = ops._q3(q)
    k_A, v_buffer = ops.as_rows(k_A), ops.as_rows(v_buffer)
    qt_hi, qt_lo = ops.absorb_q(q3, k_B, want_lo=True)
    # 8 heads of 128 under ranks 256 / 384 / 512: one workgroup serves every kv head of a split
    wide = hkv == 8 and dv == 128 and hq <= 32 and k_A.shape[-1] in (256, 384, 512) and v_buffer.stride(2) == dv
    # Everything else is register-staged: two workgroups per CU and 64-token tiles up to rank 256, one and 32 beyond (us with a plan
    # for one and 32 / for two and 64: rank 256, 64 heads on 8, batch 32 x 4000 171 / 109, batch 8 x 7001 80 / 54; rank 512 466 / 472, 210 / 218)
    splits, cap, S, plan = _plan(lens, batch, 1 if wide else hkv, kv_len, 512 if wide else k_A.shape[-1], absorbed=wide or k_A.shape[-1] > 256)
    partial, lse = ops.workspaces(batch, hq, S, dv, q.device, plan)
    ops.latent_stage1(qt_hi, qt_lo, None, (k_A, k_A.stride(0), k_A.stride(1), 0, k_A.shape[-1]), None,
                      (v_buffer, v_buffer.stride(0), v_buffer.stride(1), v_buffer.stride(2), dv),
                      partial, lse, None, splits, lens, batch, hq, hkv, kv_len, S, float(sm_scale), split_cap=cap, split_plan=plan)
    return ops.merge_stage2(partial, lse, o, None, splits, lens, batch, hq, hq, kv_len, S, split_cap=cap, split_plan=plan)


# Two passes (scores, then softmax + P.v_A) or one kernel: scores and values each run at the rate of a kernel made for them, but a third launch and
# the scores' way through memory cost 5 - 8 us.  Where the two cross is a matter of the tokens scanned (batch x kv_len) times the kv heads, each of
# which rebuilds them.  us of one kernel / two passes, 32 heads on 8 kv heads unless said:
#   values of their own: rank 256 / 256, 12288 tokens 26.4 / 27.3, 14336 29.7 / 29.7 (16 on 2: 49152 32.8 / 34.4, 65536 39.0 / 37.3); 256 / 512, 16384 35.0 / 37.1, 24576 48.9 / 43.0
#   (16 on 4: 32768 38.9 / 38.0; 16 on 2: 98304 55.5 / 55.5); 384 / 384, 16384 37.9 / 38.1, 20480 40.5 / 39.9, 24576 45.9 / 43.1 (16 on 4: 40960 41.5 / 40.0; 16 on 2: 98304 56.6 /
#   54.2); 384 / 512, 20480 42.3 / 42.0, 24576 49.3 / 45.9 (16 on 4: 49152 49.5 / 47.0; 16 on 2: 131072 74.7 / 70.0); 512 / 512, 24576 51.5 / 50.7, 30720 58.9 / 57.1 (16 on 2:
#   131072 78.6 / 78.7, 163840 94.9 / 93.6); 8 on 1, whose rows come from memory, 384 / 512, 200000 80.8 / 89.7, 300000 110 / 123; 512 / 512, 262144 108 / 104: those lines are where two passes
#   were the faster once, because calls beyond them had fp32 rotation, a scaled query and weights from the running maximum, which the one kernel has not (bf16, rank 256 / 256, 131072 tokens: 1.8e-3 from
#   float64 against 1.5e-3, peaked 2.4e-3 and 1.6e-3; queries of 65504 give NaN);
#   rank pairs without an 8-wave kernel, 512 / 384: 4096 31.8 / 33.2, 8192 45.5 / 38.8 (8 on 1: 98304 63.9 / 51.9)
#   one basis: rank 128, 8192 23.5 / 25.6, 14336 28.7 / 27.4 (16 on 2: 57344 29.9 / 29.6; 8 on 1: 131072 33.2 / 32.5); rank 192, 8192 25.9 / 27.9, 14336 32.1 / 30.3, 131072 143 / 78.7
#   (16 on 2: 57344 32.9 / 32.4; 8 on 1: 131072 36.2 / 37.8, 262144 52.9 / 55.4); rank 256 with several kv heads a workgroup one kernel, which the native layer takes before it asks, else (64 on 8, 65536 50.9 / 57.6, 163840
#   111 / 114, 262144 179 / 174; 24 on 6: 98304 58.0 / 62.9, 163840 88.1 / 88.3, 262144 140 / 129; 32 on 4: 262144 97.5 / 105; 16 on 2: 131072 39.6 / 48.5) as exact as calls were that
#   had no such kernel: even weights in bf16 3.8e-4 from float64 against 3.3e-4, peaked ones 2.1e-3 and 1.2e-3; rank 384 and 512 one kernel up to 131072 tokens (122 / 130, 142 / 161)
TWO_PASS_KEY_RANKS = (512, 384, 256)
TWO_PASS_MIN_TOKENS = 49152         # where a caller's counts are taken, whatever the kv heads; the other lines are in thirds of it
TWO_PASS_WORK = {(256, 256): 6, (256, 512): 8, (384, 384): 10, (384, 512): 10, (512, 512): 15}   # tokens x kv heads, pairs with an 8-wave kernel
TWO_PASS_WORK_ONE = {(384, 384): 14, (384, 512): 14}    # of one kv head, where that is another line
TWO_PASS_WORK_OTHER = 2
TWO_PASS_WORK_SHARED = {128: (1, 114688), 192: (2, 114688), 256: (4, 409600)}    # least kv heads, tokens x kv heads
# Key ranks up to 192 have no 8-wave kernel: two passes from this many tokens x kv heads on, and from four times as many at the ranks
# that the generic kernel is instantiated for (key rank 64, value rank 256, 1024 tokens 17.6 / 18.9, 4096 27.8 / 24.7; 16 on 4, 2048 19.7 / 20.6, 3072 22.9 / 21.7;
# 8 on 1, 8192 21.5 / 23.1, 12288 24.1 / 23.4; key rank 192, value rank 512, 4096 27.8 / 30.3, 8192 38.3 / 37.4, 16384 59.4 / 40.1; 16 on 4, 8192 28.5 / 30.2, 16384
# 38.9 / 33.7; 16 on 2, 16384 29.2 / 31.8, 32768 38.7 / 34.5).
TWO_PASS_SMALL_RANK = 192
TWO_PASS_MIN_TOKENS_SMALL = 12288
GENERIC_RANKS = (128, 192)
# A ragged batch in one kernel is scanned with the caller's counts, which may leave most of the device idle (16 heads on 2 kv heads, 8 splits
# of 7368 tokens: 84 us, two passes 29): two passes from here on, whatever the heads.
TWO_PASS_MIN_TOKENS_ASKED = 4096


def _two_pass(rank, tokens, k_B, asked=False, v_rank=512, shared=False):
    hkv = k_B.shape[1]
    if shared:
        least, work = TWO_PASS_WORK_SHARED.get(rank, (1, float("inf")))
        return hkv >= least and tokens * hkv >= work
    if rank in TWO_PASS_KEY_RANKS:
        work = TWO_PASS_WORK.get((rank, v_rank), TWO_PASS_WORK_OTHER)
        if hkv == 1:
            work = TWO_PASS_WORK_ONE.get((rank, v_rank), work)
        return tokens * hkv >= work * TWO_PASS_MIN_TOKENS // 3 or (asked and tokens >= TWO_PASS_MIN_TOKENS)
    if rank > TWO_PASS_SMALL_RANK or not ops._row_ok(k_B):
        return False
    if asked:
        return tokens >= TWO_PASS_MIN_TOKENS_ASKED
    return tokens * hkv >= TWO_PASS_MIN_TOKENS_SMALL * (4 if rank in GENERIC_RANKS else 1)


def decode_rope(q_pe, k_A, k_B, v_A, v_B, o, num_kv_splits, max_kv_splits, sm_scale, theta, sin_cos,
                pos_offset=0, kv_lens=None):
    """K = RoPE(k_A @ k_B) rebuilt and rotated in registers, V factorised."""
    ops.check_splits(num_kv_splits, max_kv_splits, q_pe.shape[0])
    if sin_cos is None and kv_lens is None and ops.USE_RECON_WORKSPACE:
        native = _lib.native()
        shared = v_A is k_A or (v_A.data_ptr() == k_A.data_ptr() and v_A.shape == k_A.shape and v_A.stride() == k_A.stride())
        two_pass = _two_pass(k_A.shape[-1], k_A.shape[0] * k_A.shape[1], k_B, v_rank=v_A.shape[-1], shared=shared)
        done = native and native.rope_decode(q_pe, k_A, k_B, v_A, v_B, o, sm_scale,
                                             ops.rope_inv_freq(q_pe.shape[-1], theta, q_pe.device), pos_offset, two_pass)
        if done is not None:
            return done
    assert v_A.shape[1] == k_A.shape[1]
    assert v_B.shape[1] == k_B.shape[1]
    batch, hq, hkv, d = _common(q_pe, k_A, k_B)
    ops.check_16bit(q_pe, k_A, k_B, v_A, v_B)
    assert d == 128, "the RoPE reconstruction kernels are built for head_dim 128"
    assert hq // hkv <= 16 and k_A.shape[-1] <= 512
    rank_v = v_A.shape[-1]
    assert rank_v == v_B.shape[2], "Rank mismatch between v_A and v_B"
    assert rank_v % 64 == 0 and rank_v <= 512
    kv_len = k_A.shape[1]
    lens = _lens(kv_lens, batch, q_pe.device)
    q3 = ops._q3(q_pe)
    k_A, v_A = ops.as_rows(k_A), ops.as_rows(v_A)
    k_B = k_B if k_B.stride(-1) == 1 else k_B.contiguous()
    inv = None
    if sin_cos is None:
        inv = ops.rope_inv_freq(d, theta, q_pe.device)
    else:
        assert sin_cos.shape == (kv_len, d), "sin_cos must be [kv_len, head_dim]"
        if sin_cos.dtype != q_pe.dtype or sin_cos.stride(-1) != 1:
            sin_cos = sin_cos.to(q_pe.dtype).contiguous()
    same_basis = (v_A.data_ptr() == k_A.data_ptr() and v_A.shape == k_A.shape and v_A.stride() == k_A.stride())
    asked = (lens is not None and batch > 1) or sin_cos is not None       # the caller's counts are taken
    scores = None
    if (not same_basis and _two_pass(k_A.shape[-1], batch * kv_len, k_B, asked, rank_v) and sin_cos is None and hq // hkv <= 8 and hq <= 32
            and rank_v in (256, 384, 512) and kv_len % 4 == 0 and ops.USE_RECON_WORKSPACE):
        try:
            scores = torch.empty((batch, hq, kv_len), dtype=torch.float32, device=q_pe.device)
        except torch.OutOfMemoryError:      # one kernel, which needs none
            pass
    if scores is not None:
        # A value basis of its own: two passes.  The scores-only form of the reconstruction kernel runs at the rate of the
        # shared-basis fused kernel (one row stream, no P.A); softmax and P.v_A then stream v_A once for all heads at HBM
        # rate.  Fused into one kernel, the second row stream costs more than the 2 x 4 bytes per score this moves.
        # the scores do not depend on how pass 1 cuts the range: one round of workgroups per CU
        S1 = ops.occupancy_splits(batch, hkv, kv_len, tile=ops.scores_tile(k_A.shape[-1], hkv, hq // hkv, batch * kv_len), waves=1)
        ops.recon_stage1(q3, k_A, k_B, None, None, None, scores, None, lens, batch, hq,
                         hkv, kv_len, S1, float(sm_scale), True, inv, int(pos_offset), None)
        S2 = ops.latent_splits(batch, 1, kv_len, rank_v, absorbed=True)
        partial, lse = ops.workspaces(batch, hq, S2, rank_v, q_pe.device)
        ops.softmax_pv_stage1(scores, v_A, partial, lse, None, lens, batch, hq, kv_len, S2, q_pe.dtype)
        return ops.merge_stage2(partial, lse, o, v_B, None, lens, batch, hq, hkv, kv_len, S2)
    if asked:
        S, splits = int(max_kv_splits), ops.as_int32_dev(num_kv_splits, batch, q_pe.device)
    else:
        S, splits = ops.decode_splits(batch, hkv, kv_len, k_A.shape[-1], same_basis), None
    partial, lse = ops.workspaces(batch, hq, S, rank_v, q_pe.device)
    ops.recon_stage1(q3, k_A, k_B, v_A, partial, lse, None, splits, lens, batch, hq, hkv, kv_len, S,
                     float(sm_scale), True, inv, int(pos_offset), sin_cos)
    return ops.merge_stage2(partial, lse, o, v_B, splits, lens, batch, hq, hkv, kv_len, S)
