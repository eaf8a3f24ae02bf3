"""Edges of the small kernels and of the dispatch rules: one parametrised test per kernel or branch, at the sizes where tiles,
remainders or ranges end, against float64 on the CPU."""
import pytest
import torch

from util import gen, max_abs

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
