"""Split-K flash decoding for grouped-query attention on plain K/V buffers.

Call surface of the reference's flash_decoding/gqa.py:339-434 (``decode_attention_fwd``), plus
  * ``kv_lens``: optional int32 ``[batch]`` of per-sequence lengths (ragged batch; the reference has
    one length, ``k_buffer.shape[1]``, for the whole batch - gqa.py:60,194);
  * ``decode_attention_fwd_v_factorized``: K plain, ``V = v_A @ v_B`` (the eager semantics of
    ``group_query_attention_factorized_v_only``, reference attention.py:202-274) as a split-K kernel
    that accumulates ``P @ v_A`` in rank space and multiplies by ``v_B`` after the merge.
Split ranges follow gqa.py:95-99 exactly; ``sm_scale`` multiplies the scores (gqa.py:122).  The caller's split counts are a
hint: a sequence is cut into what fills the device (split-K is exact under the merge), chosen on the host for a batch of one
length and per call on the device for a ragged one.
"""
from __future__ import annotations

import torch

from kernel_collections_amd import _lib, ops


# Shortest split, in tokens, that the wrappers cut a sequence into (0: the caller's splits as they are).  Split-K is exact under
# the merge, so the caller's count is a hint about parallelism and not part of the result: the wrappers choose the count that
# fills the device - for one length on the host, for a ragged batch per call on the device (equal jobs, at most one per
# workgroup the chip holds).  The caller's own counts miss it on both sides: 32 sequences of 1K .. 128K tokens in 4096-token
# splits are 315 jobs on 256 CUs (1040 us, planned: 748), 8 of up to 16K are 20 (113 us
# at no less than 1024 tokens each, planned: 52).
# At 128 tokens a job's start (about 5 us) is a third of its time; a batch too short to fill the device at that takes shorter ones
# (`split_floor` in csrc/host.cpp).  _WIDE: the all-heads forms, one workgroup per CU.
MAX_SPLIT_TOKENS = 128
MAX_SPLIT_TOKENS_WIDE = 128


def _plan(wide, lens, splits, S, batch, groups, kv_len, device, up):
    """(num_kv_splits, cap, split dimension of the workspaces, split plan on the device or None) of a call."""
    floor, per_cu = (MAX_SPLIT_TOKENS_WIDE, 1) if wide else (MAX_SPLIT_TOKENS, 2)
    if not floor:
        return ops.as_int32_dev(splits, batch, device), 0, S, None
    heads, groups = groups, 1 if wide else groups
    least = ops.split_floor(batch, groups, kv_len, per_cu, up)
    if wide and not up:
        least = ops.head_rows_floor(heads, batch * kv_len, least)
    floor = min(floor, least)
    if lens is not None and batch > 1:
        return ops.ragged_plan(lens, batch, groups, kv_len, floor, per_cu)
    S = min(ops.occupancy_splits(batch, groups, kv_len, tile=32, waves=per_cu), -(-kv_len // floor))
    return None, 0, S, None


def _prep(q, k_buffer, max_kv_splits, kv_lens):
    assert q.dim() == 3 and k_buffer.dim() == 4
    batch, num_q_heads, head_dim = q.shape
    num_kv_heads = k_buffer.shape[2]
    assert k_buffer.shape[0] == batch and k_buffer.shape[-1] == head_dim
    kv_group_num = num_q_heads // num_kv_heads
    assert kv_group_num >= 1 and num_q_heads % num_kv_heads == 0
    assert kv_group_num <= 32, "at most 32 query heads per kv head"
    assert head_dim % 32 == 0, "head_dim must be a multiple of 32"
    lens = None if kv_lens is None else ops.as_int32_dev(kv_lens, batch, q.device)
    return batch, num_q_heads, num_kv_heads, head_dim, int(max_kv_splits), lens


def decode_attention_fwd(q, k_buffer, v_buffer, o, num_kv_splits, max_kv_splits, sm_scale=1.0, *, kv_lens=None):
    """q ``[batch, Hq, d]``; k_buffer / v_buffer ``[batch, kv_len, Hkv, d]``; o ``[batch, Hq, d]`` (filled,
    returned); num_kv_splits int32 ``[batch]`` on the device; max_kv_splits int."""
    ops.check_splits(num_kv_splits, max_kv_splits, q.shape[0])
    native = _lib.native()
    done = native and native.gqa(q, k_buffer, v_buffer, None, o, sm_scale, kv_lens, MAX_SPLIT_TOKENS_WIDE, MAX_SPLIT_TOKENS)
    if done is not None:
        return done
    batch, hq, hkv, d, S, lens = _prep(q, k_buffer, max_kv_splits, kv_lens)
    ops.check_16bit(q, k_buffer, v_buffer)
    assert k_buffer.shape[-1] == v_buffer.shape[-1], "head dim of K and V must be the same"
    dv = v_buffer.shape[-1]
    assert dv % 64 == 0 and dv <= 512
    kv_len = k_buffer.shape[1]
    q3 = ops._q3(q)
    k_buffer, v_buffer = ops.as_rows(k_buffer), ops.as_rows(v_buffer)
    # 2, 4 or 8 kv heads of 128 side by side in a token row: stage 1 serves every head of a split from one workgroup (whole
    # rows through its LDS ring), so there are hkv times fewer workgroups and a split may be twice as long
    wide = (hkv in (2, 4, 8) and d == 128 and hq <= 32 and k_buffer.stride(2) == d and v_buffer.stride(2) == d
            and k_buffer.stride(1) >= hkv * d and v_buffer.stride(1) >= hkv * d
            and ops.head_rows(hkv, hq, batch, kv_len, lens is not None and batch > 1))
    splits, cap, S, plan = _plan(wide, lens, num_kv_splits, S, batch, hkv, kv_len, q.device, False)
    partial, lse = ops.workspaces(batch, hq, S, dv, q.device, plan)
    ops.latent_stage1(q3, None, None,
                      (k_buffer, k_buffer.stride(0), k_buffer.stride(1), k_buffer.stride(2), d), None,
                      (v_buffer, v_buffer.stride(0), v_buffer.stride(1), v_buffer.stride(2), dv),
                      partial, lse, None, splits, lens, batch, hq, hkv, kv_len, S, float(sm_scale), split_cap=cap,
                      split_plan=plan)
    return ops.merge_stage2(partial, lse, o, None, splits, lens, batch, hq, hq, kv_len, S, split_cap=cap, split_plan=plan)


def decode_attention_fwd_v_factorized(q, k_buffer, v_A_buffer, v_B_buffer, o, num_kv_splits, max_kv_splits,
                                      sm_scale=1.0, *, kv_lens=None):
    """K plain ``[batch, kv_len, Hkv, d]``; v_A ``[batch, kv_len, rv]``; v_B ``[batch, Hkv, rv, d]``."""
    ops.check_splits(num_kv_splits, max_kv_splits, q.shape[0])
    native = _lib.native()
    done = native and native.gqa(q, k_buffer, v_A_buffer, v_B_buffer, o, sm_scale, kv_lens, MAX_SPLIT_TOKENS_WIDE, MAX_SPLIT_TOKENS)
    if done is not None:
        return done
    batch, hq, hkv, d, S, lens = _prep(q, k_buffer, max_kv_splits, kv_lens)
    ops.check_16bit(q, k_buffer, v_A_buffer, v_B_buffer)
    rv = v_A_buffer.shape[-1]
    assert v_A_buffer.shape[1] == k_buffer.shape[1] and v_B_buffer.shape[1] == hkv and v_B_buffer.shape[2] == rv
    assert rv % 64 == 0 and rv <= 512
    kv_len = k_buffer.shape[1]
    q3 = ops._q3(q)
    k_buffer, v_A_buffer = ops.as_rows(k_buffer), ops.as_rows(v_A_buffer)
    # 2, 4 or 8 kv heads of 128 side by side in a token row: stage 1 serves every head of a split from one workgroup, and the value
    # basis (shared by the heads) is read once per token instead of once per kv head
    in_row = (hkv in (2, 4, 8) and d == 128 and rv in (256, 384, 512) and hq <= 32 and k_buffer.stride(2) == d
              and k_buffer.stride(1) >= hkv * d and v_A_buffer.stride(1) >= rv)
    # 512-wide token rows of other heads (2 x 256, 8 x 64 ...): the same form, with the block-diagonal query built here
    wide4 = not in_row and hkv * d == 512 and rv == 512 and hq <= 32 and k_buffer.stride(2) == d
    splits, cap, S, plan = _plan(in_row or wide4, lens, num_kv_splits, S, batch, hkv, kv_len, q.device, True)
    partial, lse = ops.workspaces(batch, hq, S, rv, q.device, plan)
    if wide4:
        ops.latent_stage1(ops.blockdiag_q(q3, hkv), None, None,
                          (k_buffer, k_buffer.stride(0), k_buffer.stride(1), 0, hkv * d), None,
                          (v_A_buffer, v_A_buffer.stride(0), v_A_buffer.stride(1), 0, rv),
                          partial, lse, None, splits, lens, batch, hq, 1, kv_len, S, float(sm_scale), split_cap=cap,
                          split_plan=plan)
    else:
        ops.latent_stage1(q3, None, None,
                          (k_buffer, k_buffer.stride(0), k_buffer.stride(1), k_buffer.stride(2), d), None,
                          (v_A_buffer, v_A_buffer.stride(0), v_A_buffer.stride(1), 0, rv),
                          partial, lse, None, splits, lens, batch, hq, hkv, kv_len, S, float(sm_scale), split_cap=cap,
                          split_plan=plan)
    return ops.merge_stage2(partial, lse, o, v_B_buffer, splits, lens, batch, hq, hkv, kv_len, S, split_cap=cap,
                            split_plan=plan)
