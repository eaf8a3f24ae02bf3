"""The native host layer: split counts, and that what it declines - operands that have to be copied first - still computes."""
import pytest
import torch

import oracle
from util import check_out, f32, gen

from kernel_collections_amd import _lib, ops


@pytest.mark.parametrize("batch,groups,kv_len,tile,per_cu", [
    (1, 1, 1, 32, 1), (1, 8, 33, 32, 1), (3, 8, 5000, 32, 1), (20, 8, 32768, 32, 1), (1, 1, 262144, 32, 1), (300, 2, 777, 64, 2),
    (64, 8, 131072, 32, 3), (7, 3, 4099, 64, 2)])
def test_balanced_splits(batch, groups, kv_len, tile, per_cu):
    """Every split of the chosen count holds tokens, and no other live count has a shorter slowest CU."""
    from kernel_collections_amd import _xkv_host
    cost = lambda S: -(-(-(-batch * S // 8) * groups) // (per_cu * 32)) * (-(-(32 * -(-(-(-kv_len // 32)) // S)) // tile) + 4)
    S = _xkv_host.balanced_splits(batch, groups, kv_len, tile, per_cu, 256)
    assert S >= 1 and ops.settled_splits(kv_len, S) == S
    live = sorted({ops.settled_splits(kv_len, n) for n in range(1, min(-(-kv_len // 32), 1024 * per_cu) + 1)})
    assert cost(S) <= min(cost(n) for n in live if batch * n * groups <= 8 * per_cu * 256 or n == 1)


@pytest.mark.gpu
@pytest.mark.parametrize("spoil", ["none", "key_rows", "query", "values", "lens"])
def test_declined_operands_take_the_general_path(dev, spoil):
    from kernel_collections_amd.flash_decoding import gqa
    b, hq, hkv, d, L = 2, 8, 2, 128, 300
    q, K, V = gen((b, hq, d), seed=1), gen((b, L, hkv, d), seed=2), gen((b, L, hkv, d), seed=3)
    lens = [L, 77]
    ref = oracle.ragged_apply(oracle.gqa_plain, lens, f32(q, K, V), (None, 1, 1), sm_scale=d ** -0.5)
    qd, Kd, Vd, o = q.to(dev), K.to(dev), V.to(dev), torch.zeros(b, hq, d, dtype=q.dtype, device=dev)
    kl = torch.tensor(lens, dtype=torch.int32, device=dev)
    if spoil == "key_rows":      # features not unit-stride
        Kd = torch.empty(b, L, hkv, d, 2, dtype=q.dtype, device=dev)[..., 0].copy_(Kd)
    elif spoil == "query":       # rows of a wider buffer
        qd = torch.empty(b, hq, d + 8, dtype=q.dtype, device=dev)[..., :d].copy_(qd)
    elif spoil == "values":      # rows whose starts are not 16-byte aligned
        Vd = torch.empty(b, L, hkv, d + 4, dtype=q.dtype, device=dev)[..., :d].copy_(Vd)
    elif spoil == "lens":
        kl = kl.to(torch.int64)
    args = (qd, Kd, Vd, None, o, d ** -0.5, kl, gqa.MAX_SPLIT_TOKENS_WIDE, gqa.MAX_SPLIT_TOKENS)
    assert (_lib.native().gqa(*args) is None) == (spoil != "none")
    ns = torch.ones(b, dtype=torch.int32, device=dev)
    assert gqa.decode_attention_fwd(qd, Kd, Vd, o.zero_(), ns, 1, d ** -0.5, kv_lens=kl) is o
    check_out(o, ref, spoil)


def test_split_hints_are_still_checked():
    """The counts are hints, but a count that fits no call is refused before any path is chosen."""
    from kernel_collections_amd.flash_decoding import gqa
    import kernel_collections_amd.flash_recontruction as fr
    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16)
    plain = lambda ns, n: gqa.decode_attention_fwd(z(2, 4, 128), z(2, 40, 2, 128), z(2, 40, 2, 128), z(2, 4, 128), ns, n)
    fact = lambda ns, n: fr.gqa_xKV_no_pe(z(2, 4, 128), z(2, 40, 64), z(2, 2, 64, 128), z(2, 40, 64), z(2, 2, 64, 128), z(2, 4, 128), ns, n, 1.0)
    for call in (plain, fact):
        with pytest.raises(AssertionError):
            call(torch.ones(3, dtype=torch.int32), 1)
        with pytest.raises(RuntimeError):
            call(torch.ones(2, dtype=torch.int32), 0)


def test_inverse_frequencies_follow_the_base():
    theta = torch.tensor(1e4)
    a = ops.rope_inv_freq(128, theta, torch.device("cpu"))
    theta.fill_(5e5)
    b = ops.rope_inv_freq(128, theta, torch.device("cpu"))
    assert not torch.equal(a, b) and torch.equal(b, ops.rope_inv_freq(128, 5e5, torch.device("cpu")))


def exhaustive_splits(batch, groups, kv_len, tile, per_cu, cus):
    """The search of balanced_splits over every number of splits."""
    blocks = -(-kv_len // 32)
    best, best_cost, seen = 1, 1 << 62, 0
    for want in range(1, min(blocks, 4 * per_cu * cus) + 1):
        per = -(-blocks // want)
        live = -(-blocks // per)
        if live == seen:
            continue
        seen = live
        rounds = -(-(-(-batch * live // 8) * groups) // (per_cu * (cus // 8)))
        cost = rounds * (-(-32 * per // tile) + 4)
        if cost < best_cost:
            best, best_cost = live, cost
        if rounds > 2 and batch * live * groups > 8 * per_cu * cus:
            break
    return best


def test_split_counts_of_a_growing_sequence():
    """One look-up a step in 31 of 32 steps of a decode loop, and the same counts as the search over every number of splits."""
    import random
    import time
    from kernel_collections_amd import _xkv_host
    rng = random.Random(3)
    for _ in range(300):
        args = (rng.choice([1, 2, 3, 5, 20, 64]), rng.choice([1, 2, 3, 8]), int(2 ** rng.uniform(0, 18)), rng.choice([16, 32, 64]), rng.choice([1, 2, 3]), 256)
        first = -(-args[2] // 32) * 32 - 31
        want = exhaustive_splits(*args)
        for kv_len in (args[2], first, first + 31):      # every length of a 32-token block
            assert _xkv_host.balanced_splits(args[0], args[1], kv_len, *args[3:]) == want, args
    best = 1e9
    for rep in range(5):
        t0 = time.perf_counter()
        for i in range(2048):
            _xkv_host.balanced_splits(1, 1, 131072 + 4096 * rep + i, 64, 2, 256)
        best = min(best, (time.perf_counter() - t0) / 2048)
    assert best < 4e-6, best      # 0.26 us; 15.8 with a search at every step


def test_a_library_of_another_abi_is_refused(tmp_path):
    import ctypes
    import subprocess
    from kernel_collections_amd import _xkv_host
    src, so = tmp_path / "old.c", tmp_path / "libold.so"
    src.write_text("int xkv_abi_version(void) { return 6; }\n")     # without the optional split counts and packed plans of version 7
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)])
    assert _lib.ABI_VERSION == _lib.lib().xkv_abi_version() == 7
    assert ctypes.CDLL(str(so)).xkv_abi_version() != _lib.ABI_VERSION
    with pytest.raises(RuntimeError, match="has ABI 6, the native host layer is built for 7"):
        _xkv_host.init(str(so))


def test_split_hints_of_no_number_are_refused():
    from kernel_collections_amd.flash_decoding import gqa
    import kernel_collections_amd.flash_recontruction as fr
    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16)
    for ns in (None, [1, 1]):
        with pytest.raises(TypeError):
            gqa.decode_attention_fwd(z(2, 4, 128), z(2, 40, 2, 128), z(2, 40, 2, 128), z(2, 4, 128), ns, 1)
        with pytest.raises(TypeError):
            fr.gqa_xKV_no_pe(z(2, 4, 128), z(2, 40, 64), z(2, 2, 64, 128), z(2, 40, 64), z(2, 2, 64, 128), z(2, 4, 128), ns, 1, 1.0)


@pytest.mark.parametrize("form,ring", [
    ("mla", True), ("mla_xkv_256", True), ("mla_xkv_384", True), ("mla_xkv_512", True), ("mla_xkv_192", False),
    ("cat", True), ("cat_288", False), ("one_buffer", True), ("prefix", True)])
def test_general_path_plans_for_the_kernel_that_runs(form, ring, monkeypatch):
    """One workgroup a CU and 32-token tiles where the ring kernel serves the call, two and 64 where the register-staged one does."""
    from kernel_collections_amd import _xkv_host
    from kernel_collections_amd.flash_decoding import deepseek_mla, mla, mla2

    class Planned(Exception):
        pass

    def stop(*shape_and_device):
        raise Planned(shape_and_device[2])
    monkeypatch.setattr(ops, "workspaces", stop)
    monkeypatch.setattr(_lib, "require_gpu", lambda t: None)
    b, hq, L = 8, 16, 65536
    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16)
    one = lambda *s: torch.zeros((1,) + s[1:], dtype=torch.bfloat16).expand(*s)
    k = one(b, L, 1, 288 if form == "cat_288" else 576)
    if form == "mla":
        call = lambda: mla2.mla_decode_attention_fwd(z(b, hq, 512), z(b, hq, 64), one(b, L, 1, 512), one(b, L, 1, 64))
    elif form.startswith("mla_xkv"):
        r = int(form[-3:])
        monkeypatch.setattr(ops, "absorb_q", lambda q, B, want_lo: (z(b, hq, r), z(b, hq, r)))
        call = lambda: mla2.mla_decode_attention_xKV(z(b, hq, 128), z(b, hq, 64), one(b, L, 1, r), z(b, 1, r, 128), one(b, L, 1, 64))
    elif form.startswith("cat"):
        w = k.shape[-1] // 9 * 8
        call = lambda: mla.decode_attention_fwd(z(b, hq, k.shape[-1]), k, k[..., :w], z(b, hq, w))
    elif form == "one_buffer":
        call = lambda: deepseek_mla.mla_decode_attention_fwd(z(b, hq, 576), k, k[..., :512])
    else:
        call = lambda: deepseek_mla.mla_decode_attention_fwd_pd_sep(z(b, hq, 576), k, k[..., :512], z(b, 32, 1, 576), z(b, 32, 1, 512))
    want = _xkv_host.balanced_splits(b, 1, L, 32 if ring else 64, 1 if ring else 2, ops.num_cus())
    with pytest.raises(Planned) as e:
        call()
    assert e.value.args[0] == want + (1 if form == "prefix" else 0)


@pytest.mark.parametrize("rank,hkv,tokens,two", [
    (64, 8, 1024, False), (64, 8, 4096, True), (64, 2, 4096, False), (64, 2, 12288, True), (64, 1, 8192, False), (64, 1, 12288, True),
    (128, 8, 4096, False), (128, 8, 16384, True), (192, 8, 4096, False), (192, 8, 16384, True), (192, 2, 16384, False), (192, 1, 24576, False)])
def test_two_passes_at_small_key_ranks_where_they_are_faster(rank, hkv, tokens, two):
    """Both sides as measured: a model of few kv heads fills the device later."""
    from kernel_collections_amd.flash_recontruction.fused_attention import _fused
    assert _fused._two_pass(rank, tokens, torch.zeros(1, hkv, rank, 128, dtype=torch.bfloat16)) == two


@pytest.mark.parametrize("rank,v_rank,hkv,tokens,two", [
    (256, 256, 8, 8192, False), (256, 256, 8, 12288, True), (256, 512, 8, 12288, False), (256, 512, 8, 16384, True), (256, 512, 2, 49152, False),
    (384, 384, 8, 16384, False), (384, 384, 8, 28672, True), (512, 512, 8, 28672, False), (512, 512, 8, 32768, True), (512, 384, 8, 4096, True), (512, 384, 8, 2048, False),
    (384, 384, 8, 20480, True), (384, 512, 8, 16384, False), (384, 512, 8, 24576, True), (384, 384, 2, 65536, False), (384, 384, 2, 98304, True),
    (256, 256, 1, 98303, False), (256, 256, 1, 98304, True), (384, 512, 1, 200000, False), (384, 512, 1, 229376, True), (384, 384, 1, 229375, False), (512, 512, 1, 262144, True),   # one kv head
    (256, 0, 6, 68266, False), (256, 0, 6, 68267, True), (256, 0, 8, 51200, True),     # one basis, whatever shares a workgroup
    (192, 0, 1, 262144, False), (192, 0, 2, 57344, True), (128, 0, 1, 131072, True), (256, 0, 2, 262144, False), (256, 0, 4, 102400, True), (384, 0, 8, 131072, False)])
def test_two_passes_where_they_are_faster(rank, v_rank, hkv, tokens, two):
    """Both sides as measured beside the lines; v_rank 0: one basis."""
    from kernel_collections_amd.flash_recontruction.fused_attention import _fused
    B = torch.zeros(1, hkv, rank, 128, dtype=torch.bfloat16)
    assert _fused._two_pass(rank, tokens, B, v_rank=v_rank or rank, shared=not v_rank) == two


@pytest.mark.parametrize("rank,hkv,G,tokens,pays", [
    (256, 8, 4, 12288, False), (256, 8, 4, 16384, True), (256, 8, 9, 16384, False), (256, 4, 4, 16384, False), (256, 4, 4, 32768, True), (256, 3, 4, 43000, False), (256, 3, 8, 54000, True),
    (256, 2, 8, 65536, False), (256, 2, 8, 131072, True), (256, 1, 8, 131072, False), (256, 1, 4, 524288, False), (384, 8, 4, 32768, False), (384, 1, 4, 262144, False)])
def test_scores_by_independent_waves_where_they_are_faster(rank, hkv, G, tokens, pays):
    """Both sides as measured beside the line: the fewer kv heads, the later."""
    from kernel_collections_amd import _xkv_host
    assert _xkv_host.recon_scores_pays(rank, hkv, G, tokens) == pays


@pytest.mark.parametrize("rank,hkv,L,tile", [(256, 8, 1000, 32), (256, 2, 20000, 32), (256, 4, 50000, 64), (192, 8, 1000, 64), (384, 8, 2500, 32)])
def test_scores_of_the_general_path_are_cut_for_the_kernel_that_runs(rank, hkv, L, tile, monkeypatch):
    from kernel_collections_amd import _xkv_host
    import kernel_collections_amd.flash_recontruction as fr
    given = []
    monkeypatch.setattr(ops, "recon_stage1", lambda *args: given.append(args[13]))
    monkeypatch.setattr(_lib, "require_gpu", lambda t: None)
    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16)
    fr.qAB_rope_v1(z(1, 4 * hkv, 1, 128), z(1, L, rank), z(1, hkv, rank, 128), 5e5)
    cut = lambda t: _xkv_host.balanced_splits(1, hkv, L, t, 1, ops.num_cus())
    assert given == [cut(tile)] and cut(tile) != cut(96 - tile)


@pytest.mark.parametrize("batch,hq,hkv,S,dv,d_out,launches", [
    (1, 32, 8, 128, 512, 128, 1), (1, 32, 8, 129, 512, 128, 2), (8, 32, 8, 32, 512, 128, 1), (8, 32, 8, 33, 512, 128, 2),
    (1, 32, 8, 33, 512, 1024, 2),      # two blocks of 512 columns, the splits of a head dealt out in each
    (2, 40, 1, 25, 512, 512, 1), (2, 40, 1, 26, 512, 512, 2),       # 40 heads of one kv head: groups of 20, folded five at a time
    (9, 16, 1, 27, 384, 512, 2), (8, 16, 1, 30, 512, 512, 1), (17, 16, 1, 14, 512, 512, 1), (9, 16, 1, 27, 256, 512, 1),     # column blocks of a head on two XCDs, or on one; few splits
    (7, 32, 1, 34, 384, 512, 2), (12, 32, 1, 20, 256, 512, 1), (4, 16, 1, 59, 256, 512, 2), (9, 16, 2, 28, 384, 128, 2), (9, 32, 8, 28, 512, 128, 1)])
def test_merge_takes_rows_first_by_the_native_rule(batch, hq, hkv, S, dv, d_out, launches, monkeypatch):
    calls = []

    class Library:
        def xkv_merge_stage2(self, *args):
            calls.append(args)
            return 0
    monkeypatch.setattr(ops._lib, "lib", lambda: Library())
    monkeypatch.setattr(ops, "stream_ptr", lambda t: None)
    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16)
    ops.merge_stage2(torch.zeros(1).expand(batch, hq, S, dv), torch.zeros(1).expand(batch, hq, S), z(batch, hq, d_out), z(1, hkv, dv, d_out).expand(batch, -1, -1, -1), None, None, batch, hq,
                     hkv, 32 * S, S)
    assert len(calls) == launches


@pytest.mark.parametrize("batch,groups,per_cu,jobs", [(1, 1, 1, 256), (32, 1, 1, 256), (128, 1, 1, 256), (129, 1, 1, 512), (64, 8, 2, 128),
                                                     (65, 8, 2, 192), (3, 300, 1, 6), (5, 512, 2, 10)])
def test_ragged_batches_get_two_jobs_a_sequence(batch, groups, per_cu, jobs):
    from kernel_collections_amd import _xkv_host
    assert _xkv_host.ragged_target(batch, groups, per_cu, 256) == jobs >= 2 * batch


@pytest.mark.parametrize("hq,hkv,r,tile,per_cu,groups", [
    (64, 8, 256, 64, 2, 8), (16, 2, 256, 64, 2, 2), (16, 2, 512, 32, 1, 2), (32, 8, 256, 32, 1, 1), (32, 8, 512, 32, 1, 1), (32, 8, 192, 64, 2, 8)])
def test_k_only_plans_for_the_kernel_that_runs(hq, hkv, r, tile, per_cu, groups, monkeypatch):
    from kernel_collections_amd import _xkv_host
    import kernel_collections_amd.flash_recontruction as fr

    class Planned(Exception):
        pass

    def stop(batch, hq, S, dv, device, plan=None):
        raise Planned(S)
    monkeypatch.setattr(ops, "workspaces", stop)
    monkeypatch.setattr(_lib, "require_gpu", lambda t: None)
    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16)
    monkeypatch.setattr(ops, "absorb_q", lambda q, B, want_lo: (z(8, hq, r), z(8, hq, r)))
    one = lambda *s: torch.zeros((1,) + s[1:], dtype=torch.bfloat16).expand(*s)
    args = (z(8, hq, 128), one(8, 7001, r), one(8, hkv, r, 128), one(8, 7001, hkv, 128), z(8, hq, 128), torch.ones(8, dtype=torch.int32), 1, 0.1)
    with pytest.raises(Planned) as e:
        fr.gqa_xKV_no_pe_k_only(*args)
    assert e.value.args[0] == _xkv_host.balanced_splits(8, groups, 7001, tile, per_cu, ops.num_cus())
    plans = []
    monkeypatch.setattr(ops, "plan_splits", lambda lens, counts, S, floor, target: plans.append((S, target)) or lens)
    with pytest.raises(Planned) as e:
        fr.gqa_xKV_no_pe_k_only(*args, kv_lens=torch.full((8,), 7001, dtype=torch.int32))
    target = _xkv_host.ragged_target(8, groups, per_cu, ops.num_cus())
    assert plans == [(target, target)] and e.value.args[0] == target


@pytest.mark.parametrize("batch,groups,kv_len,per_cu,up,floor", [
    (1, 1, 599, 1, False, 32), (8, 1, 1295, 1, False, 64), (8, 1, 2500, 1, False, 96), (32, 1, 1295, 1, False, 128),    # all heads a workgroup
    (1, 1, 5000, 1, True, 64), (8, 1, 1295, 1, True, 96), (3, 1, 5000, 1, True, 128),                                   # ... and up-projected
    (1, 2, 5000, 2, False, 64), (8, 2, 2500, 2, False, 128), (3, 2, 1295, 2, True, 64), (1, 2, 12000, 2, True, 128)])    # register-staged
def test_short_batches_are_cut_shorter(batch, groups, kv_len, per_cu, up, floor):
    """The fastest of 32, 64, 96, 128 and 256 tokens as measured, within 3 %."""
    from kernel_collections_amd import _xkv_host
    assert _xkv_host.split_floor(batch, groups, kv_len, per_cu, 256, up) == floor == ops.split_floor(batch, groups, kv_len, per_cu, up)


def test_short_sequences_under_many_heads_are_not_cut_below_64_tokens(monkeypatch):
    from kernel_collections_amd.flash_decoding import mla
    monkeypatch.setattr(_lib, "require_gpu", lambda t: None)
    k = torch.zeros(3, 1227, 1, 576, dtype=torch.bfloat16)
    assert mla.stage1_splits(3, 1227, mla.stage1_operands(torch.zeros(3, 64, 576, dtype=torch.bfloat16), k, k[..., :512])) == 20


def test_few_partial_rows_are_cut_to_32_tokens(monkeypatch):
    from kernel_collections_amd.flash_decoding import mla
    monkeypatch.setattr(_lib, "require_gpu", lambda t: None)
    k = torch.zeros(2, 832, 1, 576, dtype=torch.bfloat16)
    assert mla.stage1_splits(2, 832, mla.stage1_operands(torch.zeros(2, 16, 576, dtype=torch.bfloat16), k, k[..., :512])) == 26


def test_two_passes_where_the_callers_counts_are_taken():
    from kernel_collections_amd.flash_recontruction.fused_attention import _fused
    B = torch.zeros(1, 2, 192, 128, dtype=torch.bfloat16)
    assert _fused._two_pass(192, 7368, B, asked=True) and not _fused._two_pass(192, 7368, B) and not _fused._two_pass(192, 4095, B, asked=True)


def test_a_library_without_the_newer_entry_points_loads(tmp_path):
    """Of the same ABI version: prefix + tail decode has the launches of that version to take there."""
    import ctypes
    import subprocess
    from kernel_collections_amd import _xkv_host
    newer = {"xkv_absorb_q_tail", "xkv_merge_stage2_tail"}
    src, so = tmp_path / "plain.c", tmp_path / "libplain.so"
    src.write_text("".join(f"int {n}(void) {{ return {_lib.ABI_VERSION if n == 'xkv_abi_version' else 0}; }}\n" for n in _lib.EXPORTS if n not in newer))
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)])
    _lib._declare(ctypes.CDLL(str(so)))
    _lib.native()
    try:
        _xkv_host.init(str(so))
    finally:
        _xkv_host.init(_lib.LIB_PATH)


@pytest.mark.parametrize("hq,hkv,b,L,ragged,row", [
    (32, 4, 1, 4000, False, False), (32, 4, 2, 8192, False, False), (32, 4, 2, 8193, False, True), (16, 4, 2, 4000, False, False), (16, 4, 1, 8193, False, True),
    (32, 4, 2, 2048, True, False), (32, 4, 3, 1500, True, True), (16, 4, 3, 300, True, True), (32, 2, 1, 100, False, False), (32, 2, 1, 8193, False, True), (32, 2, 2, 100, True, True), (16, 2, 1, 100, False, True),
    (32, 8, 1, 100, False, True)])
def test_few_heads_are_one_row_where_that_is_faster(hq, hkv, b, L, ragged, row, monkeypatch):
    """Both sides as measured beside the rule, and the splits of the general path for the kernel that runs."""
    from kernel_collections_amd import _xkv_host
    from kernel_collections_amd.flash_decoding import gqa

    class Planned(Exception):
        pass

    def stop(batch, hq, S, dv, device, plan=None):
        raise Planned(S)
    assert ops.head_rows(hkv, hq, b, L, ragged) == row
    monkeypatch.setattr(ops, "workspaces", stop)
    monkeypatch.setattr(_lib, "require_gpu", lambda t: None)
    if ragged:
        return
    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16)
    with pytest.raises(Planned) as e:
        gqa.decode_attention_fwd(z(b, hq, 128), z(b, L, hkv, 128), z(b, L, hkv, 128), z(b, hq, 128), torch.ones(b, dtype=torch.int32), 1)
    groups, per_cu = (1, 1) if row else (hkv, 2)
    floor = ops.head_rows_floor(hkv, b * L, ops.split_floor(b, groups, L, per_cu, False))
    assert e.value.args[0] == min(_xkv_host.balanced_splits(b, groups, L, 32, per_cu, ops.num_cus()), -(-L // floor))


def test_rows_of_two_heads_have_no_split_of_one_tile():
    assert [ops.head_rows_floor(h, t, 32) for h, t in ((2, 4096), (2, 4097), (2, 8000), (4, 8000), (8, 8000))] == [32, 64, 64, 32, 32]
    assert ops.head_rows_floor(2, 9000, 128) == 128
