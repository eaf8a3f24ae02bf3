"""The native host layer as a serving program meets it: scratch of a ragged batch, and what a call does besides computing."""
import pytest
import torch

from util import check_out, gen

pytestmark = pytest.mark.gpu

BF, FP = torch.bfloat16, torch.float16


def one_long(b, L):
    return [L] + [1 + (37 * i) % 200 for i in range(1, b)]


@pytest.mark.parametrize("path", ["native", "general"])
@pytest.mark.parametrize("form", ["gqa", "v_factorized", "decode"])
def test_scratch_of_a_ragged_batch_follows_its_jobs(dev, path, form):
    """64 sequences, the longest of 32K tokens: partial rows for the jobs the batch is cut into, not for as many splits of every
    sequence as the longest one gets (2.1 million rows of 128 or 512 floats, 268 MB and more)."""
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd.flash_decoding import gqa
    b, L, hq, hkv, r = 64, 32768, 32, 8, 512
    lens = one_long(b, L)
    scale = 128 ** -0.5
    one = lambda *s, seed: gen(s, seed=seed).to(dev).expand(b, *s[1:])   # one cache for all
    q = gen((b, hq, 128), seed=1).to(dev)
    if path == "general":       # rows of a wider buffer: the native layer declines, the wrapper copies q and launches by itself
        q = torch.empty(b, hq, 136, dtype=BF, device=dev)[..., :128].copy_(q)
    kl = torch.tensor(lens, dtype=torch.int32, device=dev)
    ns = torch.full((b,), 4, dtype=torch.int32, device=dev)
    o = torch.empty(b, hq, 128, dtype=BF, device=dev)
    vB = gen((1, hkv, r, 128), std=r ** -0.5, seed=5).to(dev).expand(b, -1, -1, -1)
    if form == "gqa":
        K, V = one(1, L, hkv, 128, seed=2), one(1, L, hkv, 128, seed=3)
        run = lambda i, j, n, lens: gqa.decode_attention_fwd(q[i:j], K[i:j, :n], V[i:j, :n], o[i:j], ns[i:j], 4, scale, kv_lens=lens)
    elif form == "v_factorized":
        K, V = one(1, L, hkv, 128, seed=2), one(1, L, r, seed=3)
        run = lambda i, j, n, lens: gqa.decode_attention_fwd_v_factorized(q[i:j], K[i:j, :n], V[i:j, :n], vB[i:j], o[i:j], ns[i:j], 4, scale, kv_lens=lens)
    else:
        K, V = one(1, L, r, seed=2), one(1, L, r, seed=3)
        run = lambda i, j, n, lens: fr.gqa_xKV_no_pe(q[i:j], K[i:j, :n], vB[i:j], V[i:j, :n], vB[i:j], o[i:j], ns[i:j], 4, scale, kv_lens=lens)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    run(0, b, L, kl)
    used = torch.cuda.max_memory_allocated() - before
    # 512 jobs at most (the per-head form on 256 CUs), 32 rows of 512 floats each, and their log-sum-exps, merged rows and queries
    assert used <= 512 * hq * (r + 1) * 4 + (8 << 20), used
    got = o.clone()
    for i in (0, 1, 17, b - 1):
        run(i, i + 1, lens[i], None)
        check_out(got[i], o[i], f"sequence {i}")


def test_no_query_heads_are_refused(dev):
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd.flash_decoding import deepseek_mla, mla2
    z = lambda *s: torch.zeros(s, dtype=BF, device=dev)
    ns = torch.ones(1, dtype=torch.int32, device=dev)
    calls = [
        lambda: fr.qAB_no_pe_v1(z(1, 0, 1, 128), z(1, 40, 64), z(1, 2, 64, 128)),
        lambda: fr.qAB_rope_v1(z(1, 0, 1, 128), z(1, 40, 64), z(1, 2, 64, 128)),
        lambda: fr.gqa_xKV_no_pe(z(1, 0, 128), z(1, 40, 64), z(1, 2, 64, 128), z(1, 40, 64), z(1, 2, 64, 128), z(1, 0, 128), ns, 1, 1.0),
        lambda: deepseek_mla.mla_decode_attention_fwd_pd_sep_xKV(z(1, 0, 128), z(1, 40, 64), z(1, 1, 64, 128), z(1, 40, 64), z(1, 1, 64, 128),
                                                                 z(1, 3, 1, 128), z(1, 3, 1, 128)),
        lambda: mla2.mla_decode_attention_fwd(z(1, 0, 512), z(1, 0, 64), z(1, 40, 1, 512), z(1, 40, 1, 64)),
    ]
    for call in calls:
        with pytest.raises((AssertionError, RuntimeError, ZeroDivisionError)):
            call()


def test_out_of_memory_is_torchs_own_error(dev):
    """What a server catches to evict and try again - and the same call computes once there is room."""
    import kernel_collections_amd.flash_recontruction as fr
    L = 1 << 20
    b = 32
    q, A, B = gen((b, 32, 1, 128), seed=1).to(dev), torch.ones(1, L, 32, dtype=BF, device=dev).expand(b, -1, -1), gen((b, 8, 32, 128), seed=2).to(dev)
    call = lambda: fr.qAB_rope_v1(q, A, B, out_dtype=torch.float32)      # 4 GiB of scores
    call()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved() + (32 << 20)
    try:
        torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(dev).total_memory)
        with pytest.raises(torch.OutOfMemoryError):
            call()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert call().shape == (b, 32, 1, L)


@pytest.mark.parametrize("path,r,rv,shared", [("native", 192, 192, True), ("native", 256, 256, False), ("general", 256, 256, False)])
def test_rope_decode_without_room_for_scores_takes_one_kernel(dev, path, r, rv, shared, monkeypatch):
    """134 MB of scores where there are 32: the call needs none of them."""
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd.flash_recontruction.fused_attention import _fused
    monkeypatch.setattr(_fused, "TWO_PASS_WORK_SHARED", {192: (1, 0)})
    monkeypatch.setattr(_fused, "TWO_PASS_MIN_TOKENS", 0)
    b, hq, L = 32, 32, 32768
    t = lambda *s, std=1.0, n=0: gen(s, std=std, seed=n).to(dev)
    q, A, B = t(b, hq, 128, std=0.4, n=1), t(1, L, r, n=2).expand(b, -1, -1), t(1, 8, r, 128, std=r ** -0.5, n=3).expand(b, -1, -1, -1)
    V, vB = (A, B) if shared else (t(1, L, rv, n=4).expand(b, -1, -1), t(1, 8, rv, 128, std=rv ** -0.5, n=5).expand(b, -1, -1, -1))
    if path == "general":
        q = torch.empty(b, hq, 136, dtype=BF, device=dev)[..., :128].copy_(q)
    o, ns = torch.empty(b, hq, 128, dtype=BF, device=dev), torch.ones(b, dtype=torch.int32, device=dev)
    call = lambda: fr.gqa_xKV_rope(q, A, B, V, vB, o, ns, 1, 128 ** -0.5, 5e5)
    want = call().clone()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved() + (32 << 20)
    try:
        torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(dev).total_memory)
        check_out(call(), want, "one kernel")
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


def test_a_kernels_refusal_is_a_runtime_error(dev):
    """An error code of the C entry points keeps its text: rows wider than stage 1 serves."""
    import kernel_collections_amd.flash_recontruction as fr
    z = lambda *s: torch.zeros(s, dtype=BF, device=dev)
    with pytest.raises(RuntimeError, match="xkv_latent_stage1 failed: shape outside the built envelope .code -2") as e:
        fr.qAB_no_pe_v1(z(1, 4, 1, 128), z(1, 40, 1056), z(1, 2, 1056, 128))
    assert type(e.value) is RuntimeError


def every_call(dev, b=2, L=700, hq=8, hkv=2, r=256, seed=0):
    """name -> (call, its tensors) for each entry point of the native layer, every operand as it serves it."""
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd.flash_decoding import deepseek_mla, gqa, mla2
    t = lambda *s, std=1.0, n=0: gen(s, std=std, seed=seed + n).to(dev)
    q, A, Av = t(b, hq, 128, n=1), t(b, L, r, n=2), t(b, L, r, n=3)
    B, Bv = t(b, hkv, r, 128, std=r ** -0.5, n=4), t(b, hkv, r, 128, std=r ** -0.5, n=5)
    K, V = t(b, L, hkv, 128, n=6), t(b, L, hkv, 128, n=7)
    c, pe, qn, qr, B1 = t(b, L, 1, r, n=8), t(b, L, 1, 64, n=9), t(b, hq, 128, n=10), t(b, hq, 64, n=11), t(b, 1, r, 128, std=r ** -0.5, n=12)
    kt, vt = t(b, 33, 1, 128, n=13), t(b, 33, 1, 128, n=14)
    ns, lens = torch.full((b,), 2, dtype=torch.int32, device=dev), torch.tensor([L] + [L // 3] * (b - 1), dtype=torch.int32, device=dev)
    s = 128 ** -0.5
    new = lambda: torch.empty_like(q)
    return {
        "scores": lambda: fr.qAB_no_pe_v1(q.unsqueeze(2), A, B, sm_scale=s, out_dtype=torch.float32),
        "rope_scores": lambda: fr.qAB_rope_v1(q.unsqueeze(2), A, B, sm_scale=s, out_dtype=torch.float32),
        "decode": lambda: fr.gqa_xKV_no_pe(q, A, B, Av, Bv, new(), ns, 2, s),
        "decode_ragged": lambda: fr.gqa_xKV_no_pe(q, A, B, Av, Bv, new(), ns, 2, s, kv_lens=lens),
        "rope_decode": lambda: fr.gqa_xKV_rope(q, A, B, A, Bv, new(), ns, 2, s, 5e5),
        "rope_decode_own_values": lambda: fr.gqa_xKV_rope(q, A, B, Av, Bv, new(), ns, 2, s, 5e5),
        "gqa": lambda: gqa.decode_attention_fwd(q, K, V, new(), ns, 2, s),
        "gqa_ragged": lambda: gqa.decode_attention_fwd(q, K, V, new(), ns, 2, s, kv_lens=lens),
        "v_factorized": lambda: gqa.decode_attention_fwd_v_factorized(q, K, Av, Bv, new(), ns, 2, s),
        "mla": lambda: mla2.mla_decode_attention_fwd(q_nope(c, q), qr, c, pe, s),
        "mla_xkv": lambda: mla2.mla_decode_attention_xKV(qn, qr, c, B1, pe, s),
        "prefix_tail": lambda: deepseek_mla.mla_decode_attention_fwd_pd_sep_xKV(q, A, B1, Av, B1, kt, vt, s),
    }


def q_nope(c, q):
    return torch.cat([q, q], -1)[..., :c.shape[-1]].contiguous()


def test_launches_let_other_threads_run(dev, shim):
    """No launch of any call is made with the interpreter locked (and every call goes through the native layer)."""
    for name, call in every_call(dev).items():
        n = shim.count("shim_launches")
        call()
        assert shim.count("shim_launches") > n, name
        assert shim.count("shim_locked_calls") == 0, name
    torch.cuda.synchronize()


def general_calls(dev, L):
    """name -> a call of the wrappers' general path (operands that the native layer declines, or calls that it does not hold)."""
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd.flash_decoding import deepseek_mla, gqa, mla, mla2
    b, hq, hkv, r = 3, 8, 8, 256
    t = lambda *s, std=1.0, n=0: gen(s, std=std, seed=n).to(dev)
    wide = lambda x: torch.empty(*x.shape[:-1], x.shape[-1] + 8, dtype=BF, device=dev)[..., :x.shape[-1]].copy_(x)   # copied by the wrapper
    q, A, Av, B = wide(t(b, hq, 128, n=1)), t(b, L, r, n=2), t(b, L, r, n=3), t(b, hkv, r, 128, std=r ** -0.5, n=4)
    K, V, ns = t(b, L, hkv, 128, n=6), t(b, L, hkv, 128, n=7), torch.full((b,), 2, dtype=torch.int32, device=dev)
    kc, vc, qc, c, pe = t(b, L, 1, 576, n=8), t(b, L, 1, 512, n=9), t(b, hq, 576, std=0.1, n=10), t(b, L, 1, r, n=11), t(b, L, 1, 64, n=12)
    kt, vt, B1 = t(b, 40, 1, 576, n=13), t(b, 40, 1, 512, n=14), t(b, 1, r, 128, std=r ** -0.5, n=15)
    qr, k1, v1 = wide(t(b, hq, 64, n=16)), t(b, 70, 1, 128, n=17), t(b, 70, 1, 128, n=18)
    s, new = 128 ** -0.5, lambda w=128: torch.empty(b, hq, w, dtype=BF, device=dev)

    def cat():
        o = new(512)
        mla.decode_attention_fwd(qc, kc, vc, o)
        return o
    return {
        "scores": lambda: fr.qAB_no_pe_v1(q.unsqueeze(2), A, B, sm_scale=s),
        "rope_scores": lambda: fr.qAB_rope_v1(q.unsqueeze(2), A, B, sm_scale=s),
        "decode": lambda: fr.gqa_xKV_no_pe(q, A, B, Av, B, new(), ns, 2, s),
        "k_only": lambda: fr.gqa_xKV_no_pe_k_only(q, A, B, V, new(), ns, 2, s),
        "rope_decode_own_values": lambda: fr.gqa_xKV_rope(q, A, B, Av, B, new(), ns, 2, s, 5e5),
        "gqa": lambda: gqa.decode_attention_fwd(q, K, V, new(), ns, 2, s),
        "mla_concatenated": cat,
        "one_buffer": lambda: deepseek_mla.mla_decode_attention_fwd(qc, kc, vc),
        "prefix_tail": lambda: deepseek_mla.mla_decode_attention_fwd_pd_sep(qc, kc, vc, kt, vt),
        "prefix_tail_xkv": lambda: deepseek_mla.mla_decode_attention_fwd_pd_sep_xKV(q, A, B1, Av, B1, k1, v1, s),
        "mla": lambda: mla2.mla_decode_attention_fwd(q_nope(c, q), qr, c, pe, s),
        "mla_xkv": lambda: mla2.mla_decode_attention_xKV(q, qr, c, B1, pe, s),
    }


def test_general_calls_share_nothing_across_streams(dev, monkeypatch):
    """The first call of a size waits behind other work on its stream; the same call on another stream does not wait for it."""
    from kernel_collections_amd.flash_recontruction.fused_attention import _fused
    monkeypatch.setattr(_fused, "TWO_PASS_MIN_TOKENS", 0)
    for name, call in general_calls(dev, 900).items():
        ref = call()                     # kernels loaded; a split count of another size
        torch.cuda.synchronize()
        one, two = torch.cuda.Stream(), torch.cuda.Stream()
        calls = general_calls(dev, 3300)[name]
        torch.cuda.synchronize()
        with torch.cuda.stream(one):
            torch.cuda._sleep(20_000_000)        # about 10 ms
            first = calls()
        with torch.cuda.stream(two):
            second = calls()
        two.synchronize()
        got = second.clone()
        torch.cuda.synchronize()
        assert ref.isfinite().all() and got.isfinite().all(), name
        assert torch.equal(got, first) and torch.equal(got, calls()), name


def test_captured_calls_leave_nothing_behind(dev):
    """A call of a new size recorded into a graph does not change what the same call computes outside of it, before the graph runs."""
    for name, call in general_calls(dev, 900).items():
        call()
        big = general_calls(dev, 2500)[name]
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            captured = big()
        eager = big().clone()
        torch.cuda.synchronize()
        for _ in range(3):
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured, eager), name
            assert torch.equal(big(), eager), name


def test_calls_on_other_streams_and_threads(dev):
    """The same calls on a side stream behind other work, and from several threads with a stream each: the eager results, bit for bit."""
    import threading
    calls = [every_call(dev, seed=100 * i, L=700 + 333 * i) for i in range(4)]
    want = [{name: call() for name, call in c.items()} for c in calls]
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        torch.cuda._sleep(2_000_000)
        got = {name: call() for name, call in calls[0].items()}
    side.synchronize()
    for name, x in got.items():
        assert torch.equal(x, want[0][name]), name
    wrong = []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(5):
                    out = {name: call() for name, call in calls[i].items()}
                    torch.cuda.current_stream().synchronize()
                    wrong.extend((i, name) for name, x in out.items() if not torch.equal(x, want[i][name]))
        except Exception as e:      # noqa: BLE001 - reported by the assertion below
            wrong.append((i, e))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:5]


def test_calls_under_graph_capture(dev):
    """Each call recorded after one warm-up, replayed three times with new keys in the captured buffers' place."""
    for name in every_call(dev):
        q_sets = [every_call(dev, seed=s)[name] for s in (0, 7, 8, 9)]
        eager = [c() for c in q_sets]
        live = q_sets[0]
        tensors = lambda c: [x.cell_contents for x in c.__closure__ if isinstance(x.cell_contents, torch.Tensor) and x.cell_contents.is_floating_point()]
        static = tensors(live)
        keep = [[t.clone() for t in tensors(c)] for c in q_sets]
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = live()
        for i in (1, 2, 3):
            for dst, src in zip(static, keep[i]):
                dst.copy_(src)
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager[i]), (name, i)
            assert torch.equal(live(), eager[i]), (name, i)      # eager work between the replays


@pytest.mark.parametrize("path", ["native", "general"])
@pytest.mark.parametrize("L,lens", [(900, [0]), (900, [1]), (900, [777]), (70000, [69999]), (900, [0, 900, 31]), (9000, [33, 8999, 0, 4096])])
def test_ragged_batches_with_and_without_a_plan(dev, path, L, lens):
    """One sequence, a batch that fits the device at the shortest splits, a planned one - each sequence as alone, none as zeros."""
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd.flash_decoding import gqa
    b, hq, r = len(lens), 16, 256
    kl = torch.tensor(lens, dtype=torch.int32, device=dev)
    t = lambda *s, std=1.0, n=0: gen(s, std=std, seed=n).to(dev)
    q = t(b, hq, 128, n=1)
    if path == "general":
        q = torch.empty(b, hq, 136, dtype=BF, device=dev)[..., :128].copy_(q)
    ns, new = torch.ones(b, dtype=torch.int32, device=dev), lambda n: torch.full((n, hq, 128), float("nan"), dtype=BF, device=dev)
    for hkv in (8, 2):
        K, V, A, vA = t(b, L, hkv, 128, n=2), t(b, L, hkv, 128, n=3), t(b, L, r, n=4), t(b, L, r, n=5)
        B, vB = t(b, hkv, r, 128, std=r ** -0.5, n=6), t(b, hkv, r, 128, std=r ** -0.5, n=7)
        for name, call in {
            "gqa": lambda s, n, l: gqa.decode_attention_fwd(q[s], K[s, :n], V[s, :n], new(len(l) if l is not None else 1), ns[s], 1, 0.1, kv_lens=l),
            "v_factorized": lambda s, n, l: gqa.decode_attention_fwd_v_factorized(q[s], K[s, :n], vA[s, :n], vB[s], new(len(l) if l is not None else 1), ns[s], 1, 0.1, kv_lens=l),
            "decode": lambda s, n, l: fr.gqa_xKV_no_pe(q[s], A[s, :n], B[s], vA[s, :n], vB[s], new(len(l) if l is not None else 1), ns[s], 1, 0.1, kv_lens=l),
            "k_only": lambda s, n, l: fr.gqa_xKV_no_pe_k_only(q[s], A[s, :n], B[s], V[s, :n], new(len(l) if l is not None else 1), ns[s], 1, 0.1, kv_lens=l),
        }.items():
            got = call(slice(0, b), L, kl)
            for i, n in enumerate(lens):
                if n == 0:
                    assert (got[i] == 0).all(), (name, hkv)
                else:
                    check_out(got[i], call(slice(i, i + 1), n, None)[0], f"{name} {hkv} sequence {i}")


@pytest.mark.parametrize("hq,hkv,r,rv,per_cu", [(32, 8, 64, 0, 1), (32, 8, 128, 0, 2), (32, 8, 192, 0, 2), (32, 8, 192, 192, 1), (32, 8, 128, 64, 1),
                                                (16, 1, 256, 0, 1), (32, 8, 512, 0, 1)])
def test_one_kernel_rope_decode_is_planned_for_its_occupancy(dev, shim, hq, hkv, r, rv, per_cu):
    """Workgroups per CU of the kernel that takes scores and P.A in one, as measured beside decode_splits in csrc/host.cpp."""
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd import ops
    L = 9000
    t = lambda *s, n=0: gen(s, seed=n).to(dev)
    q, A, B = t(1, hq, 128, n=1), t(1, L, r, n=2), t(1, hkv, r, 128, n=3)
    V, vB = (t(1, L, rv, n=4), t(1, hkv, rv, 128, n=5)) if rv else (A, B)
    fr.gqa_xKV_rope(q, A, B, V, vB, torch.empty_like(q), torch.ones(1, dtype=torch.int32, device=dev), 1, 0.1, 5e5)
    assert shim.count("shim_recon_splits") == ops.occupancy_splits(1, hkv, L, tile=32, waves=per_cu)


@pytest.mark.parametrize("form", ["copied", "one_sequence"])
def test_general_rope_decode_fills_the_device(dev, form, monkeypatch):
    """The caller's two splits are a hint here too - operands to be copied first, one sequence of a given length."""
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd import ops
    L, r = 5000, 192
    t = lambda *s, std=1.0, n=0: gen(s, std=std, seed=n).to(dev)
    q, A, B = t(1, 16, 128, std=0.4, n=1), t(1, L, r, n=2), t(1, 2, r, 128, std=r ** -0.5, n=3)
    ns = torch.full((1,), 2, dtype=torch.int32, device=dev)
    want = fr.gqa_xKV_rope(q, A, B, A, B, torch.empty_like(q), ns, 2, 128 ** -0.5, 5e5)
    seen = []
    real = ops.recon_stage1
    monkeypatch.setattr(ops, "recon_stage1", lambda *a: seen.append(a[13]) or real(*a))
    kw = {}
    if form == "copied":
        q = torch.empty(1, 16, 136, dtype=BF, device=dev)[..., :128].copy_(q)
    else:
        kw = dict(kv_lens=torch.full((1,), L, dtype=torch.int32, device=dev))
    got = fr.gqa_xKV_rope(q, A, B, A, B, torch.empty(1, 16, 128, dtype=BF, device=dev), ns, 2, 128 ** -0.5, 5e5, **kw)
    assert seen == [ops.decode_splits(1, 2, L, r, True)] and seen[0] > 64
    check_out(got, want, form)


@pytest.mark.parametrize("over,launches", [("shim", 5), ("shim_tail", 3)])
@pytest.mark.parametrize("Lt", [1, 97, 1500])
def test_prefix_tail_with_and_without_the_joined_launches(dev, over, launches, Lt, request):
    """Native over a library of the ABI version alone and over one with the entry points added since, each against float64."""
    from kernel_collections_amd import _lib
    shim = request.getfixturevalue(over)
    b, hq, L, r, w = 2, 8, 700, 256, 128
    t = lambda *s, std=1.0, n=0: gen(s, std=std, seed=n).to(dev)
    a = q, kA, kB, vA, vB, kT, vT = t(b, hq, w, n=1), t(b, L, r, n=2), t(b, 1, r, w, std=r ** -0.5, n=3), t(b, L, r, n=4), t(b, 1, r, w, std=r ** -0.5, n=5), \
        t(b, Lt, 1, w, n=6), t(b, Lt, 1, w, n=7)
    got = _lib.native().prefix_tail(*a, w ** -0.5, 0.0)
    assert got is not None and shim.count("shim_launches") == launches
    q, kA, kB, vA, vB, kT, vT = (x.cpu().double() for x in a)
    k, v = torch.cat((kA @ kB[:, 0], kT[:, :, 0]), 1), torch.cat((vA @ vB[:, 0], vT[:, :, 0]), 1)
    check_out(got, (torch.softmax(q @ k.transpose(1, 2) * w ** -0.5, -1) @ v).float(), over)


def test_two_passes_over_a_library_that_lacks_their_wider_forms(dev, shim, monkeypatch):
    """Value rows of 192 and more than 32 heads came with the joined launches: without them one kernel, still native."""
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd.flash_recontruction.fused_attention import _fused
    monkeypatch.setattr(_fused, "TWO_PASS_WORK_SHARED", {x: (1, 0) for x in (128, 192, 256)})
    for hq, r in ((8, 192), (64, 256), (8, 256)):
        t = lambda *s, std=1.0, n=0: gen(s, std=std, seed=n).to(dev)
        q, A, B, ns = t(1, hq, 128, n=1), t(1, 500, r, n=2), t(1, 8, r, 128, std=r ** -0.5, n=3), torch.ones(1, dtype=torch.int32, device=dev)
        call = lambda: fr.gqa_xKV_rope(q, A, B, A, B, torch.empty_like(q), ns, 1, 0.1, 5e5)
        before = shim.count("shim_stage1")
        got = call()
        assert shim.count("shim_stage1") - before == (2 if hq <= 32 and r == 256 else 1)
        with monkeypatch.context() as m:
            m.setattr(_fused, "TWO_PASS_WORK_SHARED", {})
            check_out(got, call(), f"{hq} heads, rank {r}")
