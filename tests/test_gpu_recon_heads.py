"""recon_heads_kernel (several kv heads per workgroup) at the sizes where its periods, ring and tails end, against float64, with the LDS poisoned."""
import pytest
import torch

from util import check_out, gen

pytestmark = pytest.mark.gpu

from kernel_collections_amd import _lib, ops  # noqa: E402

BF, FP = torch.bfloat16, torch.float16
NAN = 0x7FFF7FFF


def keys_and_scores(q, A, B, off):
    """Scores [b, hq, L] of rotated reconstructed keys, in float64 on the inputs' device."""
    b, hkv, L, G = q.shape[0], B.shape[1], A.shape[1], q.shape[1] // B.shape[1]
    inv = ops.rope_inv_freq(128, 5e5, torch.device("cpu")).to(q.device)
    ang = (torch.arange(off, off + L, device=q.device).float()[:, None] * inv).double()
    k = torch.matmul(A.double().unsqueeze(1), B.double())
    lo, hi = k[..., :64], k[..., 64:]
    k = torch.cat((lo * ang.cos() - hi * ang.sin(), hi * ang.cos() + lo * ang.sin()), -1)
    s = torch.matmul(q.double().reshape(b, hkv, G, 128), k.transpose(-1, -2).contiguous())
    return s.reshape(b, hkv * G, L)


def operands(dev, dtype, b, hkv, G, L, r, stride):
    q, B = gen((b, hkv * G, 128), std=0.5, dtype=dtype, seed=1).to(dev), gen((b, hkv, r, 128), std=r ** -0.5, dtype=dtype, seed=3).to(dev)
    A = torch.full((b, L, stride), float("nan"), dtype=dtype, device=dev)[..., :r].copy_(gen((b, L, r), dtype=dtype, seed=2))
    return q, A, B


def poison():
    assert _lib.lib().xkv_poison_lds(NAN, None, torch.cuda.current_stream().cuda_stream) == 0


# S splits of n tiles each, the last one `cut` tokens short, in as many sequences as the kernel is taken for: every slot of the ring, both
# parities, tails, seeds of the angles (every 28 tiles), head slots that stay empty
S, WORKGROUPS = 24, 192
SIZES = [(r, hkv, G, n, cut) for r, hkv in ((512, 2), (512, 8), (384, 4), (256, 4)) for n, cut, G in ((1, 31, 4), (2, 1, 1), (3, 0, 3), (4, 17, 4), (5, 30, 2), (33, 5, 4))]
SIZES += [(r, 2, G, n, 9) for r in (512, 384) for n, G in ((1, 8), (6, 5), (31, 8))]


def sequences(r, hkv):
    return -(-WORKGROUPS * (4 if r == 256 else 2) // (hkv * S))


@pytest.mark.parametrize("r,hkv,G,n,cut", SIZES)
@pytest.mark.parametrize("dtype", [BF, FP])
def test_decode(dev, dtype, r, hkv, G, n, cut):
    b, L, hq, off = sequences(r, hkv), 32 * n * S - cut, hkv * G, 1000
    q, A, B = operands(dev, dtype, b, hkv, G, L, r, r + 8)
    lens = [L] + [L // 3 + 1] * (b - 1)
    kl = torch.tensor(lens, dtype=torch.int32, device=dev)
    part, lse = torch.full((b, hq, S, r), float("nan"), device=dev), torch.full((b, hq, S), float("nan"), device=dev)
    poison()
    ops.recon_stage1(q, A, B, A, part, lse, None, None, kl, b, hq, hkv, L, S, 128 ** -0.5, ops.ROPE_GROUPED, ops.rope_inv_freq(128, 5e5, q.device), off, None)
    out = torch.empty((b, hq, r), device=dev)
    ops.merge_stage2(part, lse, out, None, None, kl, b, hq, hq, L, S)
    s = keys_and_scores(q, A, B, off) * 128 ** -0.5
    for i, m in enumerate(lens):
        ref = torch.softmax(s[i, :, :m], -1) @ A[i, :m].double()
        check_out(out[i], ref, f"sequence {i}")
        # P is 16 bits wide (2^-9 or 2^-11 of it), the keys and the query were in fp16 on the way
        assert (out[i] - ref).norm() <= (4e-3 if dtype == BF else 2e-3) * ref.norm()


@pytest.mark.parametrize("r,hkv,G,n,cut", [x for x in SIZES if x[0] != 256])
@pytest.mark.parametrize("dtype,out", [(BF, torch.float32), (FP, FP)])
def test_scores(dev, dtype, out, r, hkv, G, n, cut):
    b, L, hq, off = sequences(r, hkv), 32 * n * S - cut, hkv * G, 77
    q, A, B = operands(dev, dtype, b, hkv, G, L, r, r + 16)
    ref = 0.25 * keys_and_scores(q, A, B, off)
    for _ in range(3):
        s = torch.full((b, hq, 1, L), float("nan"), dtype=out, device=dev)
        poison()
        ops.recon_stage1(q, A, B, None, None, None, s, None, None, b, hq, hkv, L, S, 0.25, ops.ROPE_GROUPED, ops.rope_inv_freq(128, 5e5, q.device), off, None)
        d = s[:, :, 0].double() - ref
        # The key and the query rounded to fp16 once each: 2.06e-4 of their size over all mantissas, together 2.9e-4; the result in fp16 as much more.  Angles in fp32
        # up to position 25000: half a unit, 2^-10 radians, at the fastest pairs, half of that on average over tokens and 1 / 64 .. of the pairs: 1e-4.
        assert d.norm() <= (3.5e-4 if out == torch.float32 else 4.2e-4) * ref.norm()
        assert d.abs().max() <= 4e-3 * ref.abs().max()      # a tile read before it is there would be of the size of the scores


@pytest.mark.parametrize("scale", [65504.0, 2.0 ** -12])
def test_scores_of_large_and_small_queries(dev, scale):
    """A rotated pair is up to 1.41 times as long as its larger feature, past fp16's largest number; a query below 6e-5 is subnormal there."""
    q, A, B = operands(dev, FP, 1, 2, 4, 6144, 512, 512)
    A *= 0.02
    q = q.sign() * scale if scale > 1 else q * scale
    s = torch.empty((1, 8, 1, 6144), device=dev)
    ops.recon_stage1(q, A, B, None, None, None, s, None, None, 1, 8, 2, 6144, 192, 1.0, ops.ROPE_GROUPED, ops.rope_inv_freq(128, 5e5, q.device), 0, None)
    ref = keys_and_scores(q, A, B, 0)
    assert (s[:, :, 0].double() - ref).norm() <= 4e-4 * ref.norm()


def test_splits_fill_the_device_once(dev, shim):
    """A call past the line is cut for workgroups of several heads, a short one and one of a single kv head for one each."""
    import kernel_collections_amd.flash_recontruction as fr
    for hkv, L, r, groups in ((8, 28672, 512, 4), (8, 28600, 512, 8), (4, 73728, 384, 2), (4, 73700, 384, 4), (8, 43008, 256, 2), (8, 43000, 256, 8), (2, 229376, 512, 1), (2, 229300, 512, 2),
                              (1, 200000, 512, 1)):
        q, A, B = operands(dev, BF, 1, hkv, 4, L, r, r)
        fr.gqa_xKV_rope(q, A, B, A, B, torch.empty_like(q), torch.ones(1, dtype=torch.int32, device=dev), 1, 0.1, 5e5)
        assert shim.count("shim_recon_splits") == ops.occupancy_splits(1, groups, L, tile=32, waves=1)


@pytest.mark.parametrize("r,hkv", [(512, 2), (384, 2), (256, 4)])
@pytest.mark.parametrize("S", [2, WORKGROUPS])                    # one kv head a workgroup, and several
@pytest.mark.parametrize("dtype,size", [(FP, 65504.0), (BF, 2.0 ** -24), (FP, 0.0)])
def test_decode_of_large_and_small_queries(dev, dtype, size, r, hkv, S):
    """As of the scores alone: a rotated pair may leave fp16's range where neither of its features does, and small ones are subnormal there."""
    L, G, off = 6144, 3, 100
    q, A, B = operands(dev, dtype, 1, hkv, G, L, r, r)
    q = q.sign() * size if size > 1 else q * size
    scale = 0.25 / size if size else 1.0
    part, lse = torch.full((1, hkv * G, S, r), float("nan"), device=dev), torch.full((1, hkv * G, S), float("nan"), device=dev)
    poison()
    ops.recon_stage1(q, A, B, A, part, lse, None, None, None, 1, hkv * G, hkv, L, S, scale, ops.ROPE_GROUPED if S > 2 else True, ops.rope_inv_freq(128, 5e5, q.device), off, None)
    out, total = torch.empty((1, hkv * G, r), device=dev), torch.empty((1, hkv * G), device=dev)
    ops.merge_stage2(part, lse, out, None, None, None, 1, hkv * G, hkv * G, L, S, total)
    s = keys_and_scores(q, A, B, off) * scale
    ref = torch.softmax(s, -1) @ A.double()
    # P is 16 bits wide (2^-9 or 2^-11 of it), the keys and the query were in fp16 on the way: 2.9e-4 of a score, in a row's sum as much at most
    assert (out - ref).norm() <= (4e-3 if dtype == BF else 2e-3) * ref.norm()
    assert (total - torch.logsumexp(s, -1)).abs().max() <= 4e-4 * max(1.0, s.abs().max().item())


@pytest.mark.parametrize("hq,hkv,L,shared", [(32, 8, 52000, True), (24, 6, 70000, True), (8, 1, 98304, False)])     # calls that scores and values apart once served, or do
def test_long_decode_of_large_queries(dev, hq, hkv, L, shared):
    import kernel_collections_amd.flash_recontruction as fr
    q, A, B = operands(dev, FP, 1, hkv, hq // hkv, L, 256, 256)
    q = q.sign() * 65504
    V = gen((1, hkv, 256, 128), std=1 / 16, dtype=FP, seed=5).to(dev)
    vA = A if shared else gen((1, L, 256), dtype=FP, seed=4).to(dev)
    o = fr.gqa_xKV_rope(q, A, B, vA, V, torch.empty(1, hq, 128, device=dev), torch.ones(1, dtype=torch.int32, device=dev), 1, 0.25 / 65504, 5e5)
    P = torch.softmax(keys_and_scores(q, A, B, 0) * (0.25 / 65504), -1)
    ref = ((P @ vA.double()).reshape(1, hkv, hq // hkv, 256) @ V.double()).reshape(1, hq, 128)
    # as above; fp32 angles up to position 70000: half a unit, 2^-8 radians, at the fastest pairs, 2.5e-4 of a score beside the 2.9e-4
    assert (o - ref).norm() <= 3e-3 * ref.norm()


def test_scores_of_decode_at_rank_256(dev):
    """Peaked rows: a split's log-sum-exp is its largest score, which the call had from a pass of its own before one kernel served it."""
    r, hkv, G, L, S, scale = 256, 4, 4, 6144, WORKGROUPS, 4.0
    q, A, B = operands(dev, BF, 1, hkv, G, L, r, r)
    part, lse = torch.empty((1, hkv * G, S, r), device=dev), torch.empty((1, hkv * G, S), device=dev)
    ops.recon_stage1(q, A, B, A, part, lse, None, None, None, 1, hkv * G, hkv, L, S, scale, ops.ROPE_GROUPED, ops.rope_inv_freq(128, 5e5, q.device), 0, None)
    s = keys_and_scores(q, A, B, 0) * scale
    err = lse - torch.logsumexp(s.reshape(1, hkv * G, S, L // S), -1)
    # The key and the query rounded to fp16 once each: 2.9e-4 of the scores' size (3072 rows: within 2 %); rotated in fp16 besides, with cosines of 16 bits, 3.9e-4
    assert err.pow(2).mean().sqrt() <= 3.2e-4 * s.pow(2).mean().sqrt()


def test_the_largest_weight_at_rank_256_is_exact(dev):
    """One token outweighs the others by e^8 and more: its weight is 1, as in a pass over given scores, however close a largest score before it came."""
    r, hkv, G, n, S, scale = 256, 4, 4, 6, WORKGROUPS, 10.0
    L = 32 * n * S
    q, A, B = operands(dev, BF, 1, hkv, G, L, r, r)
    part, lse = torch.empty((1, hkv * G, S, r), device=dev), torch.empty((1, hkv * G, S), device=dev)
    ops.recon_stage1(q, A, B, A, part, lse, None, None, None, 1, hkv * G, hkv, L, S, scale, ops.ROPE_GROUPED, ops.rope_inv_freq(128, 5e5, q.device), 0, None)
    s = (keys_and_scores(q, A, B, 0) * scale).reshape(hkv * G, S, 32 * n)
    top = s.topk(2, -1).values
    gap = top[..., 0] - top[..., 1]
    close = (gap > 8) & (gap < 14)
    ref = torch.softmax(s, -1).unsqueeze(2) @ A[0].double().reshape(S, 32 * n, r)
    err = (part[0] - ref[:, :, 0]).norm(dim=-1) / ref[:, :, 0].norm(dim=-1)
    # the others: a few e^-8, times the error of their scores, 3e-4 of 57; a weight of 1 to 2 in bf16 would be 1e-3 off
    assert close.sum() > 500 and err[close].max() <= 2e-4


def test_several_heads_where_the_splits_are_known(dev):
    """Counts or lengths on the device, splits that leave a round half empty and short calls keep one kv head a workgroup, as a factor at an odd place does."""
    r, hkv, G = 512, 8, 4

    def call(L, S, odd=False, counts=None, lens=None, rope=True):
        q, A, B = operands(dev, BF, 1, hkv, G, L, r, r)
        if odd:
            B = torch.empty(B.numel() + 4, dtype=BF, device=dev)[4:].view(B.shape).copy_(B)
        part, lse = torch.zeros((1, hkv * G, S, r), device=dev), torch.zeros((1, hkv * G, S), device=dev)
        to = lambda n: None if n is None else torch.tensor([n], dtype=torch.int32, device=dev)
        ops.recon_stage1(q, A, B, A, part, lse, None, to(counts), to(lens), 1, hkv * G, hkv, L, S, 128 ** -0.5, rope, ops.rope_inv_freq(128, 5e5, q.device), 0, None)
        return part

    one = call(28672, 64, odd=True)      # a copy of the factor: never several heads
    assert torch.equal(call(28672, 64, counts=64), one) and torch.equal(call(28672, 64, lens=28672), one)
    several = call(28672, 64, rope=ops.ROPE_GROUPED)
    assert not torch.equal(several, one) and torch.equal(call(28672, 64), several)      # one round of 256 workgroups, or two of 512
    assert torch.equal(call(28672, 64, lens=28672, rope=ops.ROPE_GROUPED), several)
    assert torch.equal(call(30720, 80), call(30720, 80, odd=True))                       # 320 in two rounds, or 640 in three
    assert torch.equal(call(20480, 64), call(20480, 64, odd=True))                       # short
