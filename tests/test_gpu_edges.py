"""Edges of the small kernels and of the dispatch rules: one parametrised test per kernel or branch, at the sizes where tiles,
remainders or ranges end, against float64 on the CPU."""
import pytest
import torch

import oracle
from util import check_out, check_scores, f32, gen, max_abs

pytestmark = pytest.mark.gpu

from kernel_collections_amd import ops  # noqa: E402

BF, FP = torch.bfloat16, torch.float16


@pytest.mark.parametrize("dtype", [BF, FP])
@pytest.mark.parametrize("b,hq,hkv,d,r", [
    (2, 32, 8, 128, 512),    # whole tiles: 4 heads of 16 rows, 64 ranks per workgroup
    (1, 3, 3, 32, 8),        # one head, one k-step, a rank below one 16-row block
    (1, 34, 2, 256, 72),     # 17 heads per kv head (a second head block of one), the last d without split features, rank remainder
    (2, 16, 1, 288, 40),     # split features with an empty wave, rank remainder
    (1, 32, 1, 512, 256),    # split features, full
    (1, 8, 2, 40, 24),       # head_dim not a multiple of 32: the scalar form
])
def test_absorb_q(dev, dtype, b, hq, hkv, d, r):
    q, B = gen((b, hq, d), dtype=dtype, seed=1), gen((b, hkv, r, d), std=d ** -0.5, dtype=dtype, seed=2)
    ref = torch.einsum("bkgd,bkrd->bkgr", q.double().reshape(b, hkv, hq // hkv, d), B.double()).reshape(b, hq, r)
    hi, lo = ops.absorb_q(q.to(dev), B.to(dev))
    # hi + lo carry twice the operand's mantissa (2 x 8 or 2 x 11 bits, at least 2^-16 of |q~| <= ~5) on top of an fp32 sum
    got = hi.double().cpu() + lo.double().cpu()
    assert max_abs(got, ref) <= 2.0 ** -16 * ref.abs().max().item()
    assert max_abs(hi, ref) <= 2.0 ** (-8 if dtype == BF else -11) * ref.abs().max().item()


@pytest.mark.parametrize("b,hq,hkv,S,live,dv,d_out", [
    (2, 8, 2, 1, 1, 64, 0),          # rows only: one split, narrowest chunk
    (1, 4, 4, 9, 9, 128, 0),         # one split past a round of eight
    (1, 2, 2, 300, 270, 512, 0),     # many splits in 64-wide chunks, dead ones at the end
    (2, 3, 1, 7, 5, 70, 0),          # rows that are not a multiple of 16 bytes
    (1, 2, 1, 40, 33, 30, 0),
    (2, 32, 8, 2, 2, 512, 128),      # up-projection: full rows, two column blocks
    (1, 5, 1, 3, 2, 192, 40),        # five heads (a second group of one), a partial column block
    (1, 24, 2, 4, 4, 256, 72),       # 12 heads per kv head, the last dv with four packets per thread
    (1, 32, 1, 1, 1, 512, 512),      # 32 heads on one factor, more head groups than fit one workgroup's LDS
    (1, 6, 2, 65, 60, 320, 128),     # many splits: rows first, then the up-projection
    (2, 3, 1, 2, 2, 70, 24),         # odd dv in the up-projecting form
])
@pytest.mark.parametrize("dtype", [BF, FP])
def test_merge(dev, dtype, b, hq, hkv, S, live, dv, d_out):
    kv_len = 32 * live                                     # 32 tokens per split: `live` of S splits hold tokens
    part = gen((b, hq, S, dv), dtype=torch.float32, seed=1)
    lse = gen((b, hq, S), std=4.0, dtype=torch.float32, seed=2)
    w = torch.softmax(lse[..., :live].double(), -1)
    ref = (w.unsqueeze(-1) * part[:, :, :live].double()).sum(2)
    part[:, :, live:], lse[..., live:] = float("nan"), float("nan")      # dead splits are never read
    vB = None
    if d_out:
        vB = gen((b, hkv, dv, d_out), std=dv ** -0.5, dtype=dtype, seed=3)
        ref = torch.einsum("bkgr,bkrd->bkgd", ref.reshape(b, hkv, hq // hkv, dv), vB.double()).reshape(b, hq, d_out)
        vB = vB.to(dev)
    out = torch.empty((b, hq, d_out or dv), dtype=torch.float32, device=dev)
    lse_out = torch.empty((b, hq), dtype=torch.float32, device=dev)
    ops.merge_stage2(part.to(dev), lse.to(dev), out, vB, ops.uniform_splits(b, S, dev), None, b, hq, hkv if d_out else hq, kv_len, S,
                     lse_out=lse_out)
    # fp32 sums of at most 300 splits and 512 ranks of unit terms, v_exp_f32 weights to 2^-21 of their value at |lse| <= 20
    assert max_abs(out, ref) <= 2e-5 * max(1.0, ref.abs().max().item())
    assert max_abs(lse_out, torch.logsumexp(lse[..., :live].double(), -1)) <= 1e-5


@pytest.mark.parametrize("dtype", [BF, FP])
@pytest.mark.parametrize("dn", [256, 384, 512])
@pytest.mark.parametrize("lens,S", [
    ([1], 1),            # one token: every row pair repeats it
    ([33], 1),           # a tile and one token
    ([640, 517], 2),     # each loader queue wraps several times; an odd end
])
def test_ring_absorbed_with_rope_features(dev, dtype, dn, lens, S):
    """The ring kernel over an absorbed query (high + low part) with 64 RoPE features behind it, ranks 256 / 384 / 512."""
    import test_gpu_ring_forms as forms
    for hq in (8, 32):
        forms.run_form(dev, dtype, hq=hq, dn=dn, lo=True, rope=True, mode="shared", dv=dn, lens=lens, S=S)


@pytest.mark.parametrize("dn,dv", [(256, 256), (256, 512), (384, 256)])
def test_ring_row_pairs_at_odd_ends(dev, dn, dv):
    """Two 512-byte rows share a load instruction: ends one token past a pair, a tile, a split."""
    import test_gpu_ring_forms as forms
    for lens, S in (([1], 1), ([31], 1), ([65, 2], 2)):
        forms.run_form(dev, BF, hq=16, dn=dn, lo=True, rope=False, mode="row", dv=dv, lens=lens, S=S)


@pytest.mark.parametrize("dtype,out", [(BF, torch.float32), (FP, FP)])
@pytest.mark.parametrize("b,hq,hkv,L,r,S,lens,off", [
    (1, 4, 1, 1, 192, 1, None, 0),              # one token: one wave works, three have no tile
    (2, 8, 2, 33, 32, 1, [33, 16], 0),          # smallest rank; a last tile of one token, a sequence of one tile
    (1, 16, 1, 2212, 192, 1, None, 131072),     # 35 steps: every buffer, angles seeded three times; 16 heads per kv head
    (1, 6, 2, 2049, 128, 3, None, 5),           # odd length (scalar stores), several splits
    (2, 3, 3, 260, 160, 4, [260, 65], 0),       # one head per kv head, splits without tokens
    (1, 8, 2, 448, 96, 1, None, 0), (1, 8, 2, 256, 64, 2, None, 0),   # whole steps only
])
def test_recon_scores_small_ranks(dev, dtype, out, b, hq, hkv, L, r, S, lens, off):
    q, A, B = gen((b, hq, 128), std=0.5, dtype=dtype, seed=1), gen((b, L, r), dtype=dtype, seed=2), \
        gen((b, hkv, r, 128), std=r ** -0.5, dtype=dtype, seed=3)
    cos, sin = oracle.rope_cos_sin(torch.arange(off, off + L), 128, 5e5)
    ref = 0.25 * oracle.qab_rope(*f32(q.unsqueeze(2), A, B), cos, sin)
    qd, Ad, Bd = q.to(dev), A.to(dev), B.to(dev)
    kl = None if lens is None else torch.tensor(lens, dtype=torch.int32, device=dev)
    got = {}
    # the same factor at an odd 8-byte place: not 16-byte packets, so the register-staged kernel
    shifted = torch.empty(B.numel() + 4, dtype=dtype, device=dev)[4:].view(B.shape).copy_(Bd)
    for name, f in (("waves", Bd), ("staged", shifted)):
        s = torch.full((b, hq, 1, L), float("nan"), dtype=out, device=dev)
        ops.recon_stage1(qd, Ad, f, None, None, None, s, ops.uniform_splits(b, S, qd.device), kl, b, hq, hkv, L, S, 0.25, True,
                         ops.rope_inv_freq(128, 5e5, qd.device), off, None)
        got[name] = s
        for i in range(b):
            n = L if lens is None else lens[i]
            check_scores(s[i, ..., :n], ref[i, ..., :n], name)
            assert s[i, ..., n:].isnan().all()      # nothing is written past a sequence


@pytest.mark.parametrize("dtype,out", [(BF, torch.float32), (FP, FP), (BF, BF)])
@pytest.mark.parametrize("b,hq,hkv,L,r,S,lens,off", [
    (1, 4, 1, 1, 256, 1, None, 0),              # one token
    (2, 8, 1, 97, 224, 1, [97, 15], 0),         # an odd number of k-steps; two steps, the last of one token; less than a tile
    (1, 5, 1, 131, 256, 1, None, 7),            # three steps: a tail of every length ...
    (1, 7, 1, 259, 256, 1, None, 0),            # ... and five: one group of groups and a tail of one
    (1, 16, 1, 1123, 224, 1, None, 131072),     # 18 steps, angles seeded twice, 16 heads per kv head
    (1, 6, 2, 2049, 384, 3, None, 5), (1, 5, 1, 2049, 384, 3, None, 5),   # two waves a tile: odd length, several splits
    (2, 3, 3, 260, 320, 4, [260, 65], 0),       # splits without tokens
    (1, 16, 2, 33, 512, 1, None, 0), (1, 8, 2, 66, 512, 1, None, 0), (1, 8, 2, 98, 448, 1, None, 0),   # two, three, four steps
    (1, 8, 2, 640, 512, 1, None, 99999),        # whole steps only, angles seeded twice
])
def test_recon_scores_large_ranks(dev, dtype, out, b, hq, hkv, L, r, S, lens, off, monkeypatch):
    if r in (384, 512):    # with a workspace the wave-specialised kernel, as at rank 256 in calls this short, without one the generic one
        test_recon_scores_small_ranks(dev, dtype, out, b, hq, hkv, L, r, S, lens, off)
        monkeypatch.setattr(ops, "USE_RECON_WORKSPACE", False)
    test_recon_scores_small_ranks(dev, dtype, out, b, hq, hkv, L, r, S, lens, off)


@pytest.mark.parametrize("dtype,out", [(BF, torch.float32), (FP, FP), (BF, BF)])
@pytest.mark.parametrize("G,S,L", [(1, 1, 4096), (4, 1, 4097), (5, 3, 4096), (8, 2, 4098)])
def test_recon_scores_rank_256(dev, dtype, out, G, S, L):
    """Ends of steps and groups where the call, by the rows it may have, is long enough for the independent waves; rows past a sequence are NaN."""
    from kernel_collections_amd import _xkv_host
    from test_gpu_recon_heads import keys_and_scores
    lens, hkv, off = [1, 97, 131, 259, 64, 1123, 65, L], 4, 131072 - 4096
    b, hq, r = len(lens), hkv * G, 256
    assert _xkv_host.recon_scores_pays(r, hkv, G, b * L)
    q, B = gen((b, hq, 128), std=0.5, dtype=dtype, seed=1).to(dev), gen((b, hkv, r, 128), std=r ** -0.5, dtype=dtype, seed=3).to(dev)
    A = gen((b, L, r), dtype=dtype, seed=2).to(dev)
    ref = 0.25 * keys_and_scores(q, A, B, off)
    for i, n in enumerate(lens):
        A[i, n:] = float("nan")
    s = torch.full((b, hq, 1, L), float("nan"), dtype=out, device=dev)
    ops.recon_stage1(q, A, B, None, None, None, s, None, torch.tensor(lens, dtype=torch.int32, device=dev), b, hq, hkv, L, S, 0.25, True, ops.rope_inv_freq(128, 5e5, q.device), off, None)
    for i, n in enumerate(lens):
        check_scores(s[i, ..., :n].cpu(), ref[i, :, None, :n].float().cpu(), f"{n} tokens")


@pytest.mark.parametrize("hkv,r", [(4, 384), (1, 320), (4, 448)])
def test_recon_scores_ends_of_two_wave_tiles(dev, hkv, r):
    """The last tile's scores meet in the LDS place of the tile four before: every number of steps from one on, each in many workgroups."""
    b, S = 1, 32
    for n in range(1, 13):        # steps of 32 tokens of a split, the last one whole or of one token
        for L in (32 * n * S, 32 * n * S - 31):
            test_recon_scores_small_ranks(dev, BF, torch.float32, b, 4 * hkv, hkv, L, r, S, None, 3)


@pytest.mark.parametrize("r,G,workspace", [(64, 16, True), (192, 4, True), (224, 1, True), (224, 16, True), (256, 9, True), (256, 16, True), (320, 4, True), (320, 8, True),
                                           (448, 5, True), (256, 4, False), (256, 8, False), (384, 4, False), (512, 8, False)])
def test_scores_of_an_exact_query(dev, r, G, workspace, monkeypatch):
    """Every rank, and calls without a workspace: no rounding but the keys' to fp16 (ranks 256, 384 and 512 with a workspace and up to 8 heads have the query's too)."""
    monkeypatch.setattr(ops, "USE_RECON_WORKSPACE", workspace)
    import kernel_collections_amd.flash_recontruction as fr
    L, hkv = 1500, 2
    for dtype in (BF, FP):
        q, A, B = gen((1, hkv * G, 1, 128), dtype=dtype, seed=1), gen((1, L, r), dtype=dtype, seed=2), gen((1, hkv, r, 128), std=r ** -0.5, dtype=dtype, seed=3)
        ang = (torch.arange(L).float()[:, None] * ops.rope_inv_freq(128, 5e5, torch.device("cpu"))).double()
        ref = oracle.qab_rope(*(t.double() for t in (q, A, B)), torch.cat((ang, ang), -1).cos(), torch.cat((ang, ang), -1).sin())
        s = fr.qAB_rope_v1(q.to(dev), A.to(dev), B.to(dev), 5e5, out_dtype=torch.float32).cpu().double()
        # rounding to 11 bits: 2^-11 / sqrt(3) of a mantissa's lowest value, 0.73 of that over all mantissas: 2.06e-4; twice the rounding is 2.9e-4
        assert (s - ref).norm() <= 2.4e-4 * ref.norm(), (dtype, ((s - ref).norm() / ref.norm()).item())


@pytest.mark.parametrize("r", [64, 192, 256])
@pytest.mark.parametrize("G", [1, 4, 5, 16])
def test_recon_scores_of_large_and_small_queries(dev, r, G):
    """A rotated pair is up to 1.41 times as long as its larger feature, past fp16's largest number; the parts of a query below 6e-5 are subnormals there."""
    L, hkv = 300, 2
    A, B = gen((1, L, r), std=0.02, dtype=FP, seed=2), gen((1, hkv, r, 128), std=r ** -0.5, dtype=FP, seed=3)
    cos, sin = oracle.rope_cos_sin(torch.arange(L), 128, 5e5)
    unit = gen((1, hkv * G, 1, 128), dtype=FP, seed=1)
    huge, tiny = unit.sign() * 65504, unit * 2.0 ** -12
    none, nan, inf = torch.zeros_like(unit), unit.clone(), unit.clone()
    nan[0, 0, 0, 3], inf[0, 0, 0, 3] = float("nan"), float("inf")
    for name, q in (("huge", huge), ("tiny", tiny), ("none", none), ("one head of a NaN", nan), ("one head of an infinity", inf)):
        ref = oracle.qab_rope(*(t.double() for t in (q, A, B)), cos.double(), sin.double())
        s = torch.empty(1, hkv * G, 1, L, dtype=torch.float32, device=dev)
        Bd = B.to(dev)
        ops.recon_stage1(q.to(dev), A.to(dev), Bd, None, None, None, s, None, None, 1, hkv * G, hkv, L, 2, 1.0, True,
                         ops.rope_inv_freq(128, 5e5, Bd.device), 0, None)
        s = s.cpu().double()
        if name.startswith("one"):
            assert not s[0, 0].isfinite().any()
            s, ref = s[:, 1:], ref[:, 1:]
        # a key rounded to fp16 (2^-11 / sqrt 12 x 2 of its size, 2.8e-4 at most), at rank 256 the query too (1.41 times that), fp32 angles
        assert (s - ref).norm() <= 4e-4 * ref.norm(), (name, ((s - ref).norm() / ref.norm()).item())


@pytest.mark.parametrize("dtype", [BF, FP])
@pytest.mark.parametrize("b,hq,hkv,L,rk,rv,off", [
    (1, 8, 2, 2049, 192, 512, 0),        # a score row past whole packets by one
    (2, 16, 2, 1027, 64, 256, 70000),    # ... by three, 8 heads per kv head
    (3, 6, 3, 700, 128, 384, 0),         # whole packets
    (1, 32, 8, 998, 384, 256, 5),        # the wide ranks' kernels, two past
    (1, 4, 1, 5, 256, 256, 0),
])
def test_two_pass_rope_decode(dev, dtype, b, hq, hkv, L, rk, rv, off, monkeypatch):
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd.flash_recontruction.fused_attention import _fused
    monkeypatch.setattr(_fused, "TWO_PASS_MIN_TOKENS", 0)
    monkeypatch.setattr(_fused, "TWO_PASS_MIN_TOKENS_SMALL", 0)
    q, kA, kB = gen((b, hq, 128), std=0.4, dtype=dtype, seed=1), gen((b, L, rk), dtype=dtype, seed=2), \
        gen((b, hkv, rk, 128), std=rk ** -0.5, dtype=dtype, seed=3)
    vA, vB = gen((b, L, rv), dtype=dtype, seed=4), gen((b, hkv, rv, 128), std=rv ** -0.5, dtype=dtype, seed=5)
    cos, sin = oracle.rope_cos_sin(torch.arange(off, off + L), 128, 5e5)
    ref = oracle.gqa_factorized_rope(*f32(q.unsqueeze(2), kA, kB, vA, vB), cos, sin, sm_scale=128 ** -0.5)[:, :, 0]
    qd, kAd, kBd, vAd, vBd = (t.to(dev) for t in (q, kA, kB, vA, vB))
    ns = torch.full((b,), 2, dtype=torch.int32, device=dev)
    two = fr.gqa_xKV_rope(qd, kAd, kBd, vAd, vBd, torch.zeros_like(qd), ns, 2, 128 ** -0.5, 5e5, pos_offset=off)
    check_out(two, ref, "two passes")
    monkeypatch.setattr(_fused, "TWO_PASS_KEY_RANKS", ())
    monkeypatch.setattr(_fused, "TWO_PASS_SMALL_RANK", 0)
    check_out(fr.gqa_xKV_rope(qd, kAd, kBd, vAd, vBd, torch.zeros_like(qd), ns, 2, 128 ** -0.5, 5e5, pos_offset=off), ref, "one kernel")


@pytest.mark.parametrize("rk,rv,batched", [(256, 256, False), (256, 384, True), (384, 512, False), (512, 384, True)])
def test_two_pass_rope_decode_of_any_factor(dev, shim_tail, rk, rv, batched, monkeypatch):
    """A factor at an odd 8-byte place: scores and values apart as with any other, whatever kernel takes the scores."""
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd.flash_recontruction.fused_attention import _fused
    monkeypatch.setattr(_fused, "TWO_PASS_MIN_TOKENS", 0)
    b, hq, hkv, L = 2, 32, 8, 8211       # rank 256: tokens x kv heads past the line from which the independent waves take the scores, over a copy of the factor
    q, kA, vA = gen((b, hq, 128), std=0.4, seed=1).to(dev), gen((b, L, rk), seed=2).to(dev), gen((b, L, rv), seed=4).to(dev)
    kB, vB = gen((b if batched else 1, hkv, rk, 128), std=rk ** -0.5, seed=3).to(dev), gen((1, hkv, rv, 128), std=rv ** -0.5, seed=5).to(dev).expand(b, -1, -1, -1)
    odd = torch.empty(kB.numel() + 4, dtype=BF, device=dev)[4:].view(kB.shape).copy_(kB).expand(b, -1, -1, -1)
    kB = kB.expand(b, -1, -1, -1)
    ns = torch.ones(b, dtype=torch.int32, device=dev)
    call = lambda B: fr.gqa_xKV_rope(q, kA, B, vA, vB, torch.empty_like(q), ns, 1, 128 ** -0.5, 5e5)
    got = call(odd)
    assert shim_tail.count("shim_stage1") == 2
    check_out(got, call(kB), "odd factor")
    s = lambda B: fr.qAB_rope_v1(q.unsqueeze(2), kA, B, 5e5, out_dtype=torch.float32).double()
    assert (s(odd) - s(kB)).norm() <= 6e-4 * s(kB).norm()      # two kernels of 2.9e-4 each, or the same


@pytest.mark.parametrize("dtype", [BF, FP])
@pytest.mark.parametrize("b,hq,hkv,L,r,shared", [
    (1, 8, 2, 2049, 192, True),          # rows of 24 lanes, two an instruction; a score row past whole packets by one
    (2, 16, 4, 1027, 128, True),         # four rows an instruction; by three
    (1, 64, 8, 998, 256, True), (1, 64, 8, 700, 256, False),   # two groups of 32 heads over the same values
    (3, 48, 4, 100, 192, True),          # 12 heads per kv head, groups of 24
    (1, 4, 1, 5, 128, True), (1, 8, 8, 33, 192, True),
])
def test_two_pass_rope_decode_of_one_basis(dev, shim_tail, dtype, b, hq, hkv, L, r, shared, monkeypatch):
    import kernel_collections_amd.flash_recontruction as fr
    from kernel_collections_amd.flash_recontruction.fused_attention import _fused
    monkeypatch.setattr(_fused, "TWO_PASS_MIN_TOKENS", 0)
    q, kA, kB = gen((b, hq, 128), std=0.4, dtype=dtype, seed=1), gen((b, L, r), dtype=dtype, seed=2), \
        gen((b, hkv, r, 128), std=r ** -0.5, dtype=dtype, seed=3)
    vA = kA if shared else gen((b, L, r), dtype=dtype, seed=4)
    vB = gen((b, hkv, r, 128), std=r ** -0.5, dtype=dtype, seed=5)
    cos, sin = oracle.rope_cos_sin(torch.arange(L), 128, 5e5)
    ref = oracle.gqa_factorized_rope(*f32(q.unsqueeze(2), kA, kB, vA, vB), cos, sin, sm_scale=128 ** -0.5)[:, :, 0]
    qd, kAd, kBd, vBd = (t.to(dev) for t in (q, kA, kB, vB))
    vAd = kAd if shared else vA.to(dev)
    ns = torch.full((b,), 2, dtype=torch.int32, device=dev)
    call = lambda: fr.gqa_xKV_rope(qd, kAd, kBd, vAd, vBd, torch.zeros_like(qd), ns, 2, 128 ** -0.5, 5e5)
    for name, work in (("two passes", 0), ("one kernel", 1 << 40)):
        monkeypatch.setattr(_fused, "TWO_PASS_WORK_SHARED", {x: (1, work) for x in (128, 192, 256)})
        monkeypatch.setattr(_fused, "TWO_PASS_KEY_RANKS", () if work else (512, 384, 256))
        before = shim_tail.count("shim_stage1")
        check_out(call(), ref, name)
        assert shim_tail.count("shim_stage1") - before == (1 if work else 2)


@pytest.mark.parametrize("lens,floor,target", [
    ([1], 32, 1),                                   # one sequence, one job
    ([0, 5, 0, 4000, 33, 0], 32, 7),                # sequences without tokens have no rows
    ([300] * 40, 128, 8),                           # more sequences than jobs: one job each
    ([7 + (613 * i) % 3000 for i in range(1100)], 128, 2048),   # several chunks of sequences
])
def test_packed_plan(dev, lens, floor, target):
    """A plan without an array of counts: every job once, whole splits first, and each sequence's first partial row."""
    b = len(lens)
    n = max(b, target)
    kl = torch.tensor(lens, dtype=torch.int32, device=dev)
    plan = ops.plan_splits(kl, None, n, floor, target).cpu().tolist()
    assert len(plan) == 3 + 2 * n + b
    count = lambda cap: sum(-(-x // cap) for x in lens)
    top = max(floor, -(-max(lens) // 32) * 32)
    cap = next((c for c in range(floor, top, 32) if count(c) <= target), top)
    live = [ops.settled_splits(x, -(-x // cap)) if x else 0 for x in lens]
    assert plan[0] == cap and plan[1] == sum(live) <= n
    assert plan[2 + 2 * n:] == [sum(live[:i]) for i in range(b + 1)]
    pairs = [(plan[2 + 2 * j], plan[3 + 2 * j]) for j in range(plan[1])]
    assert sorted(pairs) == [(i, s) for i in range(b) for s in range(live[i])]
    assert all(s == live[i] - 1 for i, s in pairs[sum(max(x - 1, 0) for x in live):])


@pytest.mark.parametrize("hq,hkv,d,rv", [
    (8, 2, 64, 0), (16, 4, 128, 0),     # register-staged kernel, several kv groups a job
    (16, 8, 128, 0), (32, 8, 128, 0),   # all heads of a job in one workgroup, values per head
    (8, 8, 128, 256), (32, 8, 128, 512),   # ... one value row for all heads, up-projected
    (6, 2, 96, 192),                    # register-staged with a shared value row, up-projected
])
def test_packed_rows(dev, hq, hkv, d, rv):
    """Stage 1 and merge over packed partial rows against the same sequences alone; sequences without tokens give zeros, as before."""
    lens = [517, 0, 1, 2048, 33, 96, 1024]
    b, L, dv, floor = len(lens), max(lens), rv or d, 64
    kl = torch.tensor(lens, dtype=torch.int32, device=dev)
    q, K = gen((b, hq, d), seed=1).to(dev), gen((b, L, hkv, d), seed=2).to(dev)
    V = gen((b, L, rv) if rv else (b, L, hkv, d), seed=3).to(dev)
    vB = gen((b, hkv, rv, 64), std=rv ** -0.5, seed=4).to(dev) if rv else None
    kop = lambda K: (K, K.stride(0), K.stride(1), K.stride(2), d)
    vop = lambda V: (V, V.stride(0), V.stride(1), 0 if rv else V.stride(2), dv)
    for target in (9, 40):
        n = max(b, target)
        plan = ops.plan_splits(kl, None, n, floor, target)
        partial, lse = (torch.full(s, float("nan"), device=dev) for s in ((hq * n, dv), (hq * n,)))
        ops.latent_stage1(q, None, None, kop(K), None, vop(V), partial, lse, None, None, kl, b, hq, hkv, L, n, d ** -0.5, split_cap=floor,
                          split_plan=plan)
        o = torch.full((b, hq, 64 if rv else d), float("nan"), dtype=torch.float32, device=dev)
        lo = torch.empty(b, hq, dtype=torch.float32, device=dev)
        ops.merge_stage2(partial, lse, o, vB, None, kl, b, hq, hkv if rv else hq, L, n, lse_out=lo, split_cap=floor, split_plan=plan)
        jobs = plan[1].item()
        assert not lse[:hq * jobs].isnan().any() and lse[hq * jobs:].isnan().all()      # every row of a job, and no other
        for i, x in enumerate(lens):
            if x == 0:
                assert (o[i] == 0).all()
                continue
            p1, l1 = ops.workspaces(1, hq, 1, dv, dev)
            ops.latent_stage1(q[i:i + 1], None, None, kop(K[i:i + 1, :x]), None, vop(V[i:i + 1, :x]), p1, l1, None, None, None, 1, hq, hkv, x, 1, d ** -0.5)
            ref = torch.empty_like(o[i:i + 1])
            ops.merge_stage2(p1, l1, ref, vB[i:i + 1] if rv else None, None, None, 1, hq, hkv if rv else hq, x, 1)
            # the softmax weights are rounded to bf16 against another running maximum: two roundings of 2^-9 of the weights' sum
            assert max_abs(o[i], ref[0]) <= 2.0 ** -7 * max(1.0, ref.abs().max().item())
            assert max_abs(lo[i], l1[0, :, 0]) <= 1e-5


def merge_c(part, lse, out, vB, S, kv_len, lse_out=None):
    """xkv_merge_stage2 itself: one launch, whatever the number of splits (ops.merge_stage2 merges the rows of many splits first)."""
    from ctypes import c_int64 as i64

    from kernel_collections_amd import _lib
    b, hq, dv = lse.shape[0], lse.shape[1], part.shape[-1]
    sv = vB.stride() if vB is not None else (0, 0, 0)
    rc = _lib.lib().xkv_merge_stage2(
        _lib.ptr(part), _lib.ptr(lse), _lib.ptr(out), _lib.ptr(vB), i64(sv[0]), i64(sv[1]), i64(sv[2]), vB.shape[-1] if vB is not None else dv,
        _lib.dtype_code(vB.dtype) if vB is not None else _lib.XKV_BF16, _lib.ptr(None), _lib.ptr(None), b, hq,
        vB.shape[1] if vB is not None else hq, kv_len, S, 0, _lib.ptr(None), dv, i64(out.stride(0)), i64(out.stride(1)),
        _lib.dtype_code(out.dtype), _lib.ptr(lse_out), i64(hq), i64(1), _lib.stream_ptr(part))
    _lib.check(rc, "xkv_merge_stage2")


@pytest.mark.parametrize("b,hq,hkv,S,live,dv,d_out,shift", [
    (1, 8, 2, 128, 128, 512, 128, 0),     # two column blocks, four groups of threads
    (1, 32, 1, 33, 29, 256, 512, 0),      # the last dv with four packets per thread, dead splits, eight column blocks
    (5, 40, 4, 97, 97, 192, 72, 0),       # ten groups and idle threads; a partial second block
    (33, 32, 8, 40, 40, 320, 200, 0),     # heads fill the chip: one workgroup for all four column blocks
    (1, 3, 1, 300, 299, 70, 24, 0),       # rows that are not a multiple of 16 bytes
    (2, 4, 1, 64, 64, 256, 64, 1),        # ... whose base is not 16-byte aligned
])
@pytest.mark.parametrize("dtype", [BF, FP])
def test_merge_of_many_splits_in_one_launch(dev, dtype, b, hq, hkv, S, live, dv, d_out, shift):
    part, lse = gen((b, hq, S, dv), dtype=torch.float32, seed=1), gen((b, hq, S), std=4.0, dtype=torch.float32, seed=2)
    w = torch.softmax(lse[..., :live].double(), -1)
    vB = gen((b, hkv, dv, d_out), std=dv ** -0.5, dtype=dtype, seed=3)
    ref = torch.einsum("bkgr,bkrd->bkgd", (w.unsqueeze(-1) * part[:, :, :live].double()).sum(2).reshape(b, hkv, hq // hkv, dv), vB.double())
    part[:, :, live:], lse[..., live:] = float("nan"), float("nan")      # dead splits are never read
    pd = torch.empty(part.numel() + shift, dtype=torch.float32, device=dev)[shift:].view(part.shape).copy_(part)
    out, lo = torch.empty((b, hq, d_out), dtype=torch.float32, device=dev), torch.empty((b, hq), dtype=torch.float32, device=dev)
    merge_c(pd, lse.to(dev), out, vB.to(dev), S, 32 * live, lo)
    # fp32 sums of at most 300 splits and 512 ranks of unit terms, v_exp_f32 weights to 2^-21 of their value at |lse| <= 20
    ref = ref.reshape(b, hq, d_out)
    assert max_abs(out, ref) <= 2e-5 * max(1.0, ref.abs().max().item())
    assert max_abs(lo, torch.logsumexp(lse[..., :live].double(), -1)) <= 1e-5


def us(call):          # device time: 20 calls in a graph
    call()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for _ in range(20):
            call()
    ev, best = [torch.cuda.Event(enable_timing=True) for _ in range(2)], 1e9
    for _ in range(10):
        ev[0].record()
        g.replay()
        ev[1].record()
        torch.cuda.synchronize()
        best = min(best, ev[0].elapsed_time(ev[1]) * 50)
    return best


def test_merge_of_many_splits_keeps_the_chip_busy(dev):
    """256 splits, up-projected: one launch that folds the splits in every column block took twice as long as merging the rows first."""
    b, hq, hkv, S, dv, d_out = 1, 32, 8, 256, 512, 128
    part, lse, mid, lo = (torch.randn(s, device=dev) for s in ((b, hq, S, dv), (b, hq, S), (b, hq, 1, dv), (b, hq)))
    vB, out = torch.randn(b, hkv, dv, d_out, device=dev).to(BF), torch.empty(b, hq, d_out, dtype=BF, device=dev)

    def rows_first():
        merge_c(part, lse, mid, None, S, 32 * S, lo)
        merge_c(mid, lo, out, vB, 1, 32)
    one, two = us(lambda: merge_c(part, lse, out, vB, S, 32 * S)), us(rows_first)
    assert one <= 1.5 * two, (one, two)


@pytest.mark.parametrize("form", ["heads", "given"])
@pytest.mark.parametrize("stride,L", [
    (1 << 31, 5),          # 2^32 bytes: a 32-bit offset between two rows is zero
    ((1 << 29) - 8, 37),   # the last stride at which two rows share a load instruction
    (1 << 29, 70),         # one past it: three tiles
])
def test_rows_far_apart(dev, form, stride, L):
    """256-wide rows of a cache whose tokens lie 1 GiB and more apart, against the same rows side by side."""
    b, hq, hkv, r = 1, 16, 8, 256
    rows = gen((b, L, r), seed=1)
    far = torch.empty(stride * (L - 1) + r, dtype=BF, device=dev).as_strided((b, L, r), (8, stride, 1))
    far.copy_(rows)
    S, ns = 2, None
    if form == "heads":        # absorbed keys under plain per-head values
        q, V = gen((b, hq, r), std=0.1, seed=2), gen((b, L, hkv, 128), seed=3)
        s = torch.einsum("bhr,blr->bhl", q.double(), rows.double())
        ref = torch.einsum("bkgl,blkd->bkgd", torch.softmax(s, -1).reshape(b, hkv, -1, L), V.double()).reshape(b, hq, 128)
        qd, lo, Vd = q.to(dev), torch.zeros_like(q).to(dev), V.to(dev)
        part, lse = ops.workspaces(b, hq, S, 128, dev)
        ops.latent_stage1(qd, lo, None, (far, 0, stride, 0, r), None, (Vd, Vd.stride(0), Vd.stride(1), 128, 128), part, lse, None, ns, None,
                          b, hq, hkv, L, S, 1.0)
    else:                      # softmax and P.V over given scores
        n = (L + 3) // 4 * 4
        s = gen((b, hq, n), std=1.0, dtype=torch.float32, seed=2)
        ref = torch.softmax(s[..., :L].double(), -1) @ rows.double()
        kl = torch.tensor([L], dtype=torch.int32, device=dev)
        part, lse = ops.workspaces(b, hq, S, r, dev)
        ops.softmax_pv_stage1(s.to(dev), far, part, lse, ns, kl, b, hq, n, S, BF)
    out = torch.empty(b, hq, ref.shape[-1], dtype=torch.float32, device=dev)
    kl = torch.tensor([L], dtype=torch.int32, device=dev)
    ops.merge_stage2(part, lse, out, None, ns, kl, b, hq, hq, n if form == "given" else L, S)
    # weights rounded to bf16: 2^-9 of values up to 4.5 each, a few of them carry the sum
    assert max_abs(out, ref) <= 2.0 ** -9 * 8


@pytest.mark.parametrize("stride,L", [(1 << 31, 5), ((1 << 29) - 8, 37), (1 << 29, 70)])
def test_value_rows_of_few_heads_far_apart(dev, stride, L):
    """Plain values of two kv heads, a 256-wide row a token, whose tokens lie 1 GiB and more apart (keys side by side)."""
    b, hq, hkv, S = 1, 16, 2, 2
    q, K, V = gen((b, hq, 128), std=0.1, seed=1), gen((b, L, hkv, 128), seed=2), gen((b, L, hkv, 128), seed=3)
    far = torch.empty(stride * (L - 1) + hkv * 128, dtype=BF, device=dev).as_strided((b, L, hkv, 128), (8, stride, 128, 1))
    far.copy_(V)
    s = torch.einsum("bkgd,blkd->bkgl", q.double().reshape(b, hkv, -1, 128), K.double())
    ref = torch.einsum("bkgl,blkd->bkgd", torch.softmax(s, -1), V.double()).reshape(b, hq, 128)
    Kd, ns = K.to(dev), None
    part, lse = ops.workspaces(b, hq, S, 128, dev)
    ops.latent_stage1(q.to(dev), None, None, (Kd, Kd.stride(0), Kd.stride(1), 128, 128), None, (far, 0, stride, 128, 128), part, lse, None, ns, None,
                      b, hq, hkv, L, S, 1.0)
    out = torch.empty(b, hq, 128, dtype=torch.float32, device=dev)
    ops.merge_stage2(part, lse, out, None, ns, None, b, hq, hq, L, S)
    assert max_abs(out, ref) <= 2.0 ** -9 * 8      # as above


@pytest.mark.parametrize("hq,hkv,b,L,ragged", [(32, 4, 1, 16384, False), (32, 4, 1, 16385, False), (12, 4, 2, 4096, False), (12, 4, 2, 4097, False), (4, 4, 3, 1, False),
                                               (32, 4, 2, 2048, True), (32, 4, 2, 2049, True), (32, 2, 1, 8192, False), (32, 2, 1, 8193, False), (16, 2, 1, 4096, False), (16, 2, 1, 4097, False),
                                               (16, 2, 1, 8001, False)])
def test_few_heads_on_both_sides_of_the_lines(dev, hq, hkv, b, L, ragged):
    """One workgroup per kv head or for all, through the native layer and the general one (a query that is not packed)."""
    from kernel_collections_amd.flash_decoding import gqa
    q, K, V = gen((b, hq, 128), std=0.3, seed=1), gen((b, L, hkv, 128), seed=2), gen((b, L, hkv, 128), seed=3)
    lens = [L - 700 * i for i in range(b)] if ragged else [L] * b
    s = torch.einsum("bkgd,blkd->bkgl", q.double().reshape(b, hkv, -1, 128), K.double())
    s.masked_fill_(torch.arange(L) >= torch.tensor(lens)[:, None, None, None], float("-inf"))
    ref = torch.einsum("bkgl,blkd->bkgd", torch.softmax(s, -1), V.double()).reshape(b, hq, 128).float()
    qd, Kd, Vd, ns = q.to(dev), K.to(dev), V.to(dev), torch.full((b,), 3, dtype=torch.int32, device=dev)
    kw = {"kv_lens": torch.tensor(lens, dtype=torch.int32, device=dev)} if ragged else {}
    wide = torch.empty(b, hq, 136, dtype=BF, device=dev)[..., :128].copy_(qd)
    for name, x in (("native", qd), ("general", wide)):
        check_out(gqa.decode_attention_fwd(x, Kd, Vd, torch.empty_like(qd), ns, 3, 1.0, **kw), ref, name)


def test_rows_of_a_tail_cost_the_prefix_scan_nothing(dev):
    """A prefix scan into a workspace with rows for a tail: workgroups without tokens would deal the others out unevenly."""
    b, hq, L, S = 16, 24, 17377, 16
    k, qn, qr = torch.randn(b, L, 1, 576, device=dev).to(BF), torch.randn(b, hq, 512, device=dev).to(BF), torch.randn(b, hq, 64, device=dev).to(BF)
    C, R = (k, k.stride(0), k.stride(1), 0, 512), (k[..., 512:], k.stride(0), k.stride(1), 0, 64)

    def scan(rows):
        part, lse = ops.workspaces(b, hq, rows, 512, dev)
        cap = -(-L // (32 * S)) * 32
        call = lambda: ops.latent_stage1(qn, None, qr, C, R, C, part, lse, None, None, None, b, hq, 1, L, rows, 0.05, split_cap=cap)
        t = us(call)
        return t, part[:, :, :S], lse[:, :, :S]
    (alone, p0, l0), (beside, p1, l1) = scan(S), scan(S + 2)
    assert torch.equal(p0, p1) and torch.equal(l0, l1)
    assert beside <= 1.2 * alone, (beside, alone)      # prefix + tail: 134 us with 18 workgroups a sequence, 94 with 16


@pytest.mark.parametrize("hq,hkv,d", [(64, 8, 128), (8, 8, 64), (32, 8, 128)])
def test_a_long_sequence_among_many_short_ones_is_cut(dev, hq, hkv, d):
    """As many sequences as a round of workgroups holds jobs: the longest one is not left to one workgroup per kv head."""
    from kernel_collections_amd.flash_decoding import gqa
    for b in (64, 256):
        L = 8192
        kl = torch.tensor([L] + [64] * (b - 1), dtype=torch.int32, device=dev)
        q, K = torch.randn(b, hq, d, device=dev).to(BF), torch.randn(1, L, hkv, d, device=dev).to(BF).expand(b, -1, -1, -1)
        o, ns = torch.empty_like(q), torch.ones(b, dtype=torch.int32, device=dev)
        kl64 = torch.full_like(kl, 64)
        many = us(lambda: gqa.decode_attention_fwd(q, K, K, o, ns, 1, 0.1, kv_lens=kl))
        alone = us(lambda: gqa.decode_attention_fwd(q[:1], K[:1], K[:1], o[:1], ns[:1], 1, 0.1, kv_lens=kl[:1]))
        short = us(lambda: gqa.decode_attention_fwd(q, K, K, o, ns, 1, 0.1, kv_lens=kl64))
        # one call for both costs no more than twice the two calls; left whole, the long one took 250 us beside 40 + 30
        assert many <= 2 * (alone + short), (b, many, alone, short)


@pytest.mark.parametrize("dtype", [BF, FP])
@pytest.mark.parametrize("b,hq,L,Lt,r,rv,w,dv,cap", [
    (1, 8, 40, 1, 256, 256, 128, 128, 0.0),       # one token in the tail
    (2, 16, 300, 31, 512, 512, 512, 512, 0.0),    # less than a tile
    (1, 32, 700, 33, 384, 384, 512, 512, 30.0),   # two splits, the last of one token; two head blocks
    (1, 3, 64, 1024, 64, 192, 32, 64, 0.0),       # 32 splits of a tile; few heads, narrow rows
    (2, 40, 900, 1057, 256, 384, 256, 320, 5.0),  # 34 tiles: 17 splits of two; two groups of 20 heads
    (1, 16, 33000, 1500, 512, 512, 512, 512, 0.0),   # many prefix splits: their rows are merged first
])
def test_prefix_tail_in_one_merge(dev, dtype, b, hq, L, Lt, r, rv, w, dv, cap):
    """Absorption and tail in one launch, prefix and tail in one merge, against attention over the concatenation in float64."""
    from kernel_collections_amd import _lib
    scale = w ** -0.5
    q, kA, kB = gen((b, hq, w), dtype=dtype, seed=1).to(dev), gen((b, L, r), dtype=dtype, seed=2).to(dev), gen((b, 1, r, w), std=r ** -0.5, dtype=dtype, seed=3).to(dev)
    vA, vB = gen((b, L, rv), dtype=dtype, seed=4).to(dev), gen((b, 1, rv, dv), std=rv ** -0.5, dtype=dtype, seed=5).to(dev)
    kT, vT = gen((b, Lt, 1, w), dtype=dtype, seed=6).to(dev), gen((b, Lt, 1, dv), dtype=dtype, seed=7).to(dev)
    kT[:, -1, 0] = q[:, 0] * 2                    # the tail's last token has the largest weight of a head
    got = _lib.native().prefix_tail(q, kA, kB, vA, vB, kT, vT, scale, cap)
    assert got is not None and got.dtype == dtype
    q, kA, kB, vA, vB, kT, vT = (t.cpu().double() for t in (q, kA, kB, vA, vB, kT, vT))
    k, v = torch.cat((kA @ kB[:, 0], kT[:, :, 0]), 1), torch.cat((vA @ vB[:, 0], vT[:, :, 0]), 1)
    s = torch.einsum("bhd,bld->bhl", q, k) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    ref = torch.einsum("bhl,bld->bhd", s.softmax(-1), v)
    check_out(got, ref.float(), "prefix + tail")
