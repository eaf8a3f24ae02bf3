"""Factors in every layout that the kernels which hold them in registers read: as they are where they are 16-byte packets, else by a copy."""
import pytest
import torch

from util import gen

pytestmark = pytest.mark.gpu

from kernel_collections_amd import _lib, ops  # noqa: E402
from test_gpu_recon_heads import NAN, keys_and_scores  # noqa: E402

BF, FP = torch.bfloat16, torch.float16


def laid_out(B, how):
    """`B` [b, hkv, r, 128] with the strides of a layout; what lies between its rows is NaN."""
    b, hkv, r, d = B.shape
    if how == "whole":
        return B.contiguous()
    if how == "rank first":              # [b, r, hkv, 128]: a factor as it is learnt
        return B.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
    if how == "one for all sequences":
        return B[:1].contiguous().expand(b, hkv, r, d)
    pad, at = {"wide rows": (16, 8), "rows of no packets": (2, 0), "rows that start anywhere": (8, 3)}[how]
    buf = torch.full((b, hkv, r, d + pad), float("nan"), dtype=B.dtype, device=B.device)
    buf[..., at:at + d] = B
    return buf[..., at:at + d]


LAYOUTS = ["rank first", "one for all sequences", "wide rows", "rows of no packets", "rows that start anywhere"]


@pytest.mark.parametrize("how", LAYOUTS)
@pytest.mark.parametrize("rk,rv,G,dtype", [(512, 0, 4, BF), (384, 0, 8, FP), (256, 0, 2, BF), (512, 512, 4, FP), (384, 512, 8, BF), (384, 384, 1, FP), (256, 256, 4, BF), (256, 512, 3, FP)])
def test_decode_over_any_layout_of_the_factor(dev, rk, rv, G, dtype, how):
    """rv 0: one basis.  Bit-equal to the call over a contiguous factor, whatever the LDS held before; the first, against float64."""
    b, hkv, S = 2, 3, 2
    L, hq = 32 * 5 * S - 7, hkv * G
    q, A = gen((b, hq, 128), std=0.5, dtype=dtype, seed=1).to(dev), gen((b, L, rk), dtype=dtype, seed=2).to(dev)
    B = gen((1 if how == LAYOUTS[1] else b, hkv, rk, 128), std=rk ** -0.5, dtype=dtype, seed=3).to(dev).expand(b, hkv, rk, 128)
    V = gen((b, L, rv), dtype=dtype, seed=4).to(dev) if rv else A

    def call(factor):
        part, lse = torch.full((b, hq, S, V.shape[2]), float("nan"), device=dev), torch.full((b, hq, S), float("nan"), device=dev)
        assert _lib.lib().xkv_poison_lds(NAN, None, torch.cuda.current_stream().cuda_stream) == 0
        ops.recon_stage1(q, A, factor, V, part, lse, None, None, None, b, hq, hkv, L, S, 128 ** -0.5, True, ops.rope_inv_freq(128, 5e5, q.device), 9, None)
        return part, lse

    part, lse = call(laid_out(B, "whole"))
    other, lse2 = call(laid_out(B, how))
    assert torch.equal(part, other) and torch.equal(lse, lse2)
    out = torch.empty((b, hq, V.shape[2]), device=dev)
    ops.merge_stage2(part, lse, out, None, None, None, b, hq, hq, L, S)
    ref = torch.softmax(keys_and_scores(q, A, B, 9) * 128 ** -0.5, -1) @ V.double()
    # P is 16 bits wide (2^-9 or 2^-11 of it); two rank halves of a key are rounded to fp16 and rotated there
    assert (out - ref).norm() <= (4e-3 if dtype == BF else 2e-3) * ref.norm()


@pytest.mark.parametrize("how", LAYOUTS)
@pytest.mark.parametrize("r,hkv,G,dtype", [(512, 2, 8, BF), (384, 4, 3, FP), (256, 4, 4, BF)])
def test_several_heads_over_any_layout_of_the_factor(dev, r, hkv, G, dtype, how):
    """Splits cut for several kv heads a workgroup: whole packets bit-equal to the call over a contiguous factor, others by the kernel of one head a workgroup over a copy."""
    b, S, off = 2, 8, 9
    L, hq = 32 * 5 * S - 7, hkv * G
    q, A = gen((b, hq, 128), std=0.5, dtype=dtype, seed=1).to(dev), gen((b, L, r), dtype=dtype, seed=2).to(dev)
    B = gen((1 if how == LAYOUTS[1] else b, hkv, r, 128), std=r ** -0.5, dtype=dtype, seed=3).to(dev).expand(b, hkv, r, 128)

    def call(factor, rope):
        part, lse = torch.full((b, hq, S, r), float("nan"), device=dev), torch.full((b, hq, S), float("nan"), device=dev)
        s = torch.full((b, hq, 1, L), float("nan"), device=dev)
        for values, out in ((A, None), (None, s)):
            assert _lib.lib().xkv_poison_lds(NAN, None, torch.cuda.current_stream().cuda_stream) == 0
            ops.recon_stage1(q, A, factor, values, part, lse, out, None, None, b, hq, hkv, L, S, 128 ** -0.5, rope, ops.rope_inv_freq(128, 5e5, q.device), off, None)
        return part, lse, s

    part, lse, s = call(laid_out(B, how), ops.ROPE_GROUPED)
    other = call(laid_out(B, "whole"), ops.ROPE_GROUPED if how in LAYOUTS[:3] else True)
    assert all(torch.equal(x, y) for x, y in zip((part, lse, s), other))
    out = torch.empty((b, hq, r), device=dev)
    ops.merge_stage2(part, lse, out, None, None, None, b, hq, hq, L, S)
    ref = keys_and_scores(q, A, B, off) * 128 ** -0.5
    # the key and the query rounded to fp16 once each, 2.9e-4 of the scores' size; P is 16 bits wide (2^-9 or 2^-11 of it)
    assert (s[:, :, 0] - ref).norm() <= 3.5e-4 * ref.norm()
    ref = torch.softmax(ref, -1) @ A.double()
    assert (out - ref).norm() <= (4e-3 if dtype == BF else 2e-3) * ref.norm()


@pytest.mark.parametrize("how", LAYOUTS)
@pytest.mark.parametrize("r,G", [(512, 5), (384, 4), (256, 8), (256, 1)])
@pytest.mark.parametrize("L", [65, 24000])     # rank 256: on both sides of the line from which recon_scores_kernel takes it (143360 tokens x kv heads for three)
def test_scores_over_any_layout_of_the_factor(dev, r, G, L, how):
    b, hkv = 2, 3
    q, A = gen((b, hkv * G, 1, 128), dtype=FP, seed=1).to(dev), gen((b, L, r), std=0.2, dtype=FP, seed=2).to(dev)
    B = gen((1 if how == LAYOUTS[1] else b, hkv, r, 128), std=r ** -0.5, dtype=FP, seed=3).to(dev).expand(b, hkv, r, 128)
    import kernel_collections_amd.flash_recontruction as fr
    s = fr.qAB_rope_v1(q, A, laid_out(B, "whole"), 5e5, out_dtype=torch.float32)
    assert torch.equal(s, fr.qAB_rope_v1(q, A, laid_out(B, how), 5e5, out_dtype=torch.float32))
    ref = keys_and_scores(q[:, :, 0], A, B, 0)
    # the key and the query rounded to fp16 once each: 2.9e-4 of the scores' size; fp32 angles up to position 24000, 1e-4
    assert (s[:, :, 0].double() - ref).norm() <= 3.5e-4 * ref.norm()


@pytest.mark.parametrize("r", [256, 384, 512])
@pytest.mark.parametrize("G", [1, 4, 8])
def test_scores_of_large_and_small_queries(dev, r, G):
    """A rotated pair is up to 1.41 times as long as its larger feature, past fp16's largest number; a query below 6e-5 is subnormal there."""
    L, hkv = 300, 2
    A, B = gen((1, L, r), std=0.02, dtype=FP, seed=2).to(dev), gen((1, hkv, r, 128), std=r ** -0.5, dtype=FP, seed=3).to(dev)
    unit = gen((1, hkv * G, 128), dtype=FP, seed=1).to(dev)
    for q in (unit.sign() * 65504, unit * 2.0 ** -12, unit * 0):
        s = torch.empty((1, hkv * G, 1, L), device=dev)
        ops.recon_stage1(q, A, B, None, None, None, s, None, None, 1, hkv * G, hkv, L, 2, 1.0, True, ops.rope_inv_freq(128, 5e5, q.device), 0, None)
        ref = keys_and_scores(q, A, B, 0)
        assert (s[:, :, 0].double() - ref).norm() <= 3.5e-4 * ref.norm()
